"""The few-rows forward (csrc/rows_kernel.h): decoding steps and short prefills, at the edges of its 16-row tiles, 32-key
tiles, wave and chunk splits, against the oracle's generic attention; results and row statistics."""
import ctypes as C
import math

import pytest
import torch

from flashlight_amd import _ffi, ops
from oracle.attention import alibi_slopes
from tests.conftest import assert_parity

DEV = "cuda"


def _taken(B, Hq, Hkv, Lq, Lk, D, **kw):
    """(whether the call goes to the few-rows kernel, scratch bytes it asks for)"""
    q, k = torch.empty(B, Hq, Lq, D, dtype=torch.bfloat16), torch.empty(B, Hkv, Lk, D, dtype=torch.bfloat16)
    a = dict(scale=None, mask_kind=0, window=0, prefix=0, doc_ids=None, alibi_heads=0, softcap=0.0, biases=(), gate=None,
             diff=False, lambda_full=0.0, attended_dump=None)
    a.update(kw)
    lib = _ffi.load_library()
    p, _ = _ffi._fill_params(lib, q, k, k, q, Hq, Hkv, **a)
    n = C.c_uint64()
    return bool(lib.fl_attn_rows_plan(C.byref(p), C.byref(n))), n.value


def test_which_calls_the_few_rows_kernel_takes():
    assert _taken(1, 32, 8, 1, 32768, 128)[0] and _taken(1, 32, 8, 1, 32768, 128)[1] > 0   # decoding, cut into chunks
    assert _taken(64, 32, 8, 1, 1000, 64) == (True, 0)          # enough workgroups without chunks
    assert not _taken(1, 8, 8, 1, 128, 64)[0]                   # too short to matter
    assert _taken(2, 8, 8, 512, 512, 64, mask_kind=_ffi.MASK_CAUSAL) == (True, 0)
    assert not _taken(4, 16, 16, 4096, 4096, 128)[0]
    assert not _taken(1, 1, 2, 1, 1000, 64)[0] and not _taken(1, 3, 2, 1, 1000, 64)[0]   # (asked before the call is refused)
    # more than 32 rows against many keys: few workgroups without chunks
    for shape in ((1, 32, 8, 9, 32768, 128), (1, 8, 8, 64, 65536, 128), (1, 8, 8, 128, 65536, 64), (2, 8, 2, 40, 5000, 128)):
        assert _taken(*shape)[0] and _taken(*shape)[1] > 0, shape
    assert _taken(1, 8, 8, 64, 1024, 64) == (True, 0) and _taken(1, 1, 1, 4096, 4096, 64, mask_kind=_ffi.MASK_CAUSAL) == (True, 0)


def test_which_calls_the_front_end_cuts_into_chunks():
    """The tile kernel over chunks of the keys, or the few-rows kernel: the estimate of host.cpp at shapes where the two
    measured far apart, and the forms that cannot be cut."""
    _ffi.load_library()

    def chunks(B, Hq, Hkv, Lq, Lk, D, longer=0):
        q, k = torch.empty(B, Hq, Lq, D, dtype=torch.bfloat16), torch.empty(B, Hkv, Lk + longer, D, dtype=torch.bfloat16)[:, :, :Lk]
        return _ffi._host.key_chunks(q, k, k)

    for shape, n in (((1, 8, 8, 64, 32768, 128), 64), ((1, 8, 8, 64, 65536, 128), 64), ((1, 8, 8, 512, 65536, 128), 16),
                     ((1, 1, 1, 4096, 65536, 128), 16), ((4, 8, 8, 64, 8192, 64), 16), ((1, 24, 24, 1000, 16384, 128), 4),
                     ((1, 16, 16, 200, 16384, 32), 16), ((1, 4, 4, 128, 16384, 256), 32)):
        assert chunks(*shape) == (n, True), shape
    for shape in ((1, 32, 8, 1, 32768, 128), (1, 8, 8, 64, 4096, 128), (1, 2, 2, 48, 32768, 128), (5, 16, 16, 40, 4096, 64)):
        assert chunks(*shape)[0] > 1 and not chunks(*shape)[1], shape          # the few-rows kernel is the sooner one
    assert chunks(1, 8, 8, 64, 4095, 128)[0] == 0 and chunks(2, 8, 8, 64, 8200, 128)[0] == 0     # short; no divisor
    assert chunks(1, 8, 8, 64, 65536, 128, longer=8) == (64, True) and chunks(2, 8, 8, 64, 65536, 128, longer=8)[0] == 0
    assert chunks(4, 16, 16, 4096, 4096, 128)[0] == 0


CASES = [  # B, Hq, Hkv, Lq, Lk, D
    (1, 4, 4, 1, 129, 64), (2, 8, 2, 1, 257, 128), (1, 8, 1, 2, 545, 64), (1, 32, 2, 1, 600, 128), (1, 17, 1, 1, 4097, 64),
    (3, 8, 8, 1, 2047, 128), (33, 8, 8, 1, 1000, 64), (64, 16, 8, 1, 200, 128), (72, 16, 16, 1, 161, 64),
    (1, 2, 2, 65, 65, 64), (1, 3, 3, 100, 100, 128), (1, 4, 2, 255, 255, 64), (1, 8, 8, 511, 513, 64), (2, 6, 2, 300, 300, 64),
    (1, 2, 1, 129, 1000, 128), (1, 16, 16, 257, 257, 64),
    (1, 8, 2, 24, 4500, 128), (2, 4, 2, 33, 4099, 128), (1, 3, 3, 70, 4200, 64), (1, 2, 2, 300, 4096, 64), (1, 16, 4, 16, 8200, 128),
    (1, 1, 1, 520, 4111, 128), (2, 8, 8, 40, 1041, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("shape", CASES)
def test_few_rows_against_the_oracle(shape, fp16):
    B, Hq, Hkv, Lq, Lk, D = shape
    dt = torch.float16 if fp16 else torch.bfloat16
    g = torch.Generator().manual_seed(sum(shape))
    q = torch.randn(B, Hq, Lq, D, generator=g).to(dt)
    longer = torch.randn(2, B, Lk + 24, Hkv, D, generator=g).to(dt)   # caches in longer, sequence-major buffers
    k, v = longer[0, :, 8:8 + Lk].transpose(1, 2), longer[1, :, 16:16 + Lk].transpose(1, 2)
    dev = longer.cuda()
    kd, vd = dev[0, :, 8:8 + Lk].transpose(1, 2), dev[1, :, 16:16 + Lk].transpose(1, 2)
    pos_q, pos_k = torch.arange(Lq)[:, None], torch.arange(Lk)[None]
    row = torch.randn(B, 1, 1, Lk, generator=g)
    row[..., 3:Lk // 3] = float("-inf")
    slopes = alibi_slopes(Hq).view(1, Hq, 1, 1)
    cases = [("plain", {}, None, None, None),
             ("causal", dict(mask_kind=_ffi.MASK_CAUSAL), pos_k > pos_q, None, None),
             ("soft-cap + ALiBi", dict(softcap=4.0, alibi_heads=Hq), None, slopes * (pos_k - pos_q), 4.0),
             ("row bias", dict(biases=[(row.to(dt).cuda(), 1)]), None, row.to(dt).float(), None),
             ("fp32 row bias", dict(biases=[(row[:1].contiguous().cuda(), B)]), None, row[:1], None)]
    if Lq == Lk:
        cases += [("window", dict(mask_kind=_ffi.MASK_SLIDING, window=33), (pos_k > pos_q) | (pos_q - pos_k > 33), None, None),
                  ("prefix", dict(mask_kind=_ffi.MASK_PREFIX_LM, prefix=40), (pos_k > pos_q) & (pos_k >= 40), None, None)]
    G = Hq // Hkv
    kf, vf = (t.float().repeat_interleave(G, 1) for t in (k, v))
    for name, kw, masked, bias, cap in cases:
        lse = torch.empty(B, Hq, Lq, dtype=torch.float32, device=DEV)
        out = _ffi.attn_fwd(q.cuda(), kd, vd, lse=lse, **kw)
        s = q.float() @ kf.transpose(-1, -2) / math.sqrt(D)
        s = cap * torch.tanh(s / cap) if cap else s
        s = s + bias if bias is not None else s
        s = s.masked_fill(masked, float("-inf")) if masked is not None else s
        assert_parity(out, torch.softmax(s, -1).nan_to_num(0.0) @ vf, f"{shape} {name}")
        want = torch.logsumexp(s, -1) / math.log(2.0)
        assert (lse.cpu() - want).abs().max().item() < 1e-2, (shape, name)
        assert_parity(ops.dispatch(q.cuda(), kd, vd, **kw), torch.softmax(s, -1).nan_to_num(0.0) @ vf, f"{shape} {name} (front end)")


@pytest.mark.gpu
def test_rows_without_keys_and_extreme_logits():
    g = torch.Generator().manual_seed(5)
    q = torch.randn(2, 8, 1, 128, generator=g).to(torch.bfloat16).cuda()
    k, v = (torch.randn(2, 2, 3000, 128, generator=g).to(torch.bfloat16).cuda() for _ in range(2))
    for fill in (float("-inf"), -1e9):
        none = torch.full((2, 1, 1, 3000), fill, dtype=torch.bfloat16, device=DEV)
        lse = torch.zeros(2, 8, 1, dtype=torch.float32, device=DEV)
        assert torch.count_nonzero(_ffi.attn_fwd(q, k, v, biases=[(none, 1)], lse=lse)) == 0
        assert torch.isinf(lse).all()
    k[:, :, 1500:] *= 60.0   # the maximum jumps by hundreds of nats half way through the keys
    want = torch.nn.functional.scaled_dot_product_attention(q.float().cpu(), k.float().cpu(), v.float().cpu(), enable_gqa=True)
    assert_parity(ops.dispatch(q, k, v), want, "jump")


@pytest.mark.gpu
def test_the_workspace_is_scratch_only_when_the_caller_says_so():
    """A parameter struct with a workspace that holds something (a document call's prepared lists), used for a decoding
    step that would cut its keys into chunks: the workspace keeps its bytes unless FL_FLAG_SCRATCH gives it away."""
    g = torch.Generator().manual_seed(6)
    q = torch.randn(1, 8, 1, 64, generator=g).to(torch.bfloat16).cuda()
    k, v = (torch.randn(1, 2, 9000, 64, generator=g).to(torch.bfloat16).cuda() for _ in range(2))
    want = torch.nn.functional.scaled_dot_product_attention(q.float().cpu(), k.float().cpu(), v.float().cpu(), enable_gqa=True)
    lib, out, n = _ffi.load_library(), torch.empty_like(q), C.c_uint64()
    p, _ = _ffi._fill_params(lib, q, k, v, out, 8, 2, None, 0, 0, 0, None, 0, 0.0, (), None, False, 0.0, None)
    assert lib.fl_attn_rows_plan(C.byref(p), C.byref(n)) and n.value
    ws = torch.full((n.value,), 0x5A, dtype=torch.uint8, device=DEV)
    p.workspace, p.workspace_bytes = ws.data_ptr(), n.value
    for flags in (0, _ffi.FLAG_SCRATCH):
        p.flags = flags
        _ffi._launch_on(q.device, lib.fl_attn_fwd, p)
        assert_parity(out, want, f"flags {flags}")
        assert bool((ws == 0x5A).all()) == (not flags)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 32, 32, 100, 300, 128), (1, 9, 3, 1400, 333, 64), (3, 2, 2, 130, 77, 32), (1, 4, 4, 200, 500, 256),
                                   (2, 40, 40, 130, 64, 64)])
def test_results_in_fp32_are_what_the_16_bit_results_round(shape):
    """FL_FLAG_F32_RESULT, for partial results that are merged: the same numbers before their rounding."""
    B, Hq, Hkv, Lq, Lk, D = shape
    g = torch.Generator().manual_seed(sum(shape))
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(torch.bfloat16).cuda() for h, n in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    row = torch.randn(B, 1, 1, Lk, generator=g).cuda()
    for kw in ({}, dict(softcap=5.0), dict(mask_kind=_ffi.MASK_CAUSAL), dict(biases=[(row, 1)])):
        assert not _taken(*shape, **kw)[0]   # (the few-rows kernel rounds against other maxima)
        wide = torch.full((B, Hq, Lq, D), float("nan"), dtype=torch.float32, device=DEV)
        assert torch.equal(_ffi.attn_fwd(q, k, v, out=wide, **kw).to(torch.bfloat16), _ffi.attn_fwd(q, k, v, **kw)), kw
    with pytest.raises(_ffi.FlashlightError, match="fp32"):
        _ffi.attn_fwd(q, k, v, out=wide, gate=torch.zeros(B, Hq, Lq, D, dtype=torch.bfloat16, device=DEV))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 8, 8, 64, 16384, 128), (1, 8, 8, 48, 9003, 128), (2, 8, 8, 130, 8192, 64), (1, 8, 2, 24, 4500, 64)])
def test_chunks_of_the_keys_replay_from_a_graph(shape):
    """More than 32 rows against many keys, by either way of cutting the keys, captured and replayed on new operands."""
    B, Hq, Hkv, Lq, Lk, D = shape
    g = torch.Generator(device=DEV).manual_seed(Lk)
    q, k, v = (torch.randn(B, h, n, D, generator=g, device=DEV).to(torch.bfloat16) for h, n in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops.dispatch(q, k, v)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.dispatch(q, k, v)
    for _ in range(3):
        q.copy_(torch.randn(q.shape, generator=g, device=DEV))
        v.mul_(-0.5)
        graph.replay()
        torch.cuda.synchronize()
        eager = ops.dispatch(q, k, v)
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    G = Hq // Hkv
    kf, vf = (t.float().cpu().repeat_interleave(G, 1) for t in (k, v))
    assert_parity(eager, torch.softmax(q.float().cpu() @ kf.transpose(-1, -2) / math.sqrt(D), -1) @ vf, str(shape))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 8, 8, 1, 1024, 128), (1, 32, 8, 1, 2048, 128), (1, 2, 2, 1, 4096, 64), (1, 8, 8, 48, 4096, 128),
                                   (1, 32, 8, 1, 32768, 128)])
def test_infinite_values_stay_in_their_columns(shape):
    """An infinite value anywhere in the cache makes its column infinite and nothing else, whichever chunk of the keys holds it and
    however many chunks the merge has."""
    B, Hq, Hkv, Lq, Lk, D = shape
    g = torch.Generator().manual_seed(sum(shape))
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(torch.bfloat16) for h, n in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    assert _taken(*shape)[0] and _taken(*shape)[1] > 0   # cut into chunks
    w = torch.softmax(q.float() @ k.float().repeat_interleave(Hq // Hkv, 1).transpose(-1, -2) / math.sqrt(D), -1)
    assert w.min() > 1e-30                               # (no weight is zero in any of the types it goes through)
    v[:, :, 0, 0], v[:, :, Lk // 2 + 5, 1], v[:, :, Lk - 1, 2], v[:, :, Lk - 1, D - 1] = (math.inf, -math.inf, math.inf, -math.inf)
    want = w @ v.float().repeat_interleave(Hq // Hkv, 1)
    out = ops.dispatch(q.cuda(), k.cuda(), v.cuda()).float().cpu()
    assert torch.equal(out.isinf(), want.isinf()) and torch.equal(out[want.isinf()], want[want.isinf()])
    assert_parity(out.masked_fill(out.isinf(), 0).to(torch.bfloat16), want.masked_fill(want.isinf(), 0), str(shape))
