"""The shared-bias stripe forward (csrc/stripe_kernel.h): lengths at the edges of its 64-key waves and 32-row blocks, against the
fp32 oracle; fp32 operands; rows that attend nothing or whose logits are large; which calls take it."""
import ctypes as C
import math

import pytest
import torch

import oracle as O
from flashlight_amd import _ffi
from tests.test_abi import good_params

DEV = "cuda"


def params(S=250, D=32, H=4, **kw):
    p = good_params(D=D)
    p.B, p.Hq, p.Hkv, p.Lq, p.Lk = 12, H, H, S, S
    p.q_strides[:] = p.k_strides[:] = p.v_strides[:] = p.o_strides[:] = (S * H * D, D, H * D, 1)
    p.bias[0], p.bias_batch_div[0] = 0x60000, 6
    p.bias_strides[0][:] = (H * S * S, S * S, S, 1)
    for n, v in kw.items():
        setattr(p, n, v)
    return p


def test_which_calls_the_stripe_forward_takes():
    takes = lambda p: _ffi.plan(p)["streaming"] == 2  # noqa: E731
    lse = 0x90000
    assert takes(params()) and takes(params(S=250, D=64)) and takes(params(S=511)) and takes(params(S=256, lse=lse))
    assert _ffi.plan(params(S=256))["streaming"] == 1                     # no statistics: the streaming kernel
    assert not takes(params(S=320, lse=lse)) and not takes(params(S=256, D=64, lse=lse)) and not takes(params(S=3))
    assert not takes(params(S=513)) and not takes(params(D=128)) and not takes(params(softcap=3.0)) and not takes(params(Hkv=2))
    assert not takes(params(mask_kind=_ffi.MASK_CAUSAL))
    p = params(S=320, lse=lse)
    p.bias_dtype[0] = _ffi.FL_F32                                         # the general kernel does not stage it
    assert takes(p)
    p = params()
    p.bias_batch_div[0] = 1                                               # a bias per batch entry is not shared
    p.bias_strides[0][0] = 0
    assert not takes(p)
    p = params()
    p.o_strides[2] += 4                                                   # results leave in 16-byte stores
    assert not takes(p)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("S", [4, 31, 33, 63, 65, 97, 130, 193, 255, 257, 321, 385, 449, 510, 511])
def test_edges_against_the_oracle(S, D):
    g = torch.Generator().manual_seed(S + D)
    H, N = 2, 5
    for dt, bias_dt, row_dt, gated in ((torch.bfloat16, torch.bfloat16, None, True), (torch.float16, torch.float16, torch.float16, False),
                                       (torch.bfloat16, torch.float32, torch.float32, True)):
        mk = lambda *s: torch.randn(*s, generator=g).to(dt)  # noqa: E731
        q, k, v, gate = (mk(N, S, H, D) for _ in range(4))
        pair = torch.randn(1, H, S, S, generator=g).to(bias_dt)
        row = None
        if row_dt is not None:
            row = torch.where(torch.rand(N, 1, 1, S, generator=g) < 0.2, -6e4, 0.0).to(row_dt)
            row[..., 0] = 0
        dev = [t.to(DEV).transpose(1, 2) for t in (q, k, v, gate)]
        biases = [(pair.to(DEV), N)] + ([(row.to(DEV), 1)] if row is not None else [])
        lse = torch.empty(N, H, S, device=DEV)
        out = _ffi.attn_fwd(*dev[:3], biases=biases, gate=dev[3] if gated else None, lse=lse)
        ref = O.attention_evoformer(q.float(), k.float(), v.float(), [pair.float()] + ([row.float()] if row is not None else []),
                                    **({"gate": gate.float()} if gated else {})).transpose(1, 2)
        # rounded weights and result: 2^-9 / sqrt 3 (bf16) or 2^-12 / sqrt 3 each, of terms that do not add up coherently
        rel = ((out.float().cpu() - ref).norm() / ref.norm()).item()
        assert rel < (3e-3 if dt == torch.bfloat16 else 4e-4), (S, D, dt, rel)
        s = q.double().transpose(1, 2) @ k.double().permute(0, 2, 3, 1) / D ** 0.5 + pair.double() + (row.double() if row is not None else 0)
        want = torch.logsumexp(s, -1) / math.log(2.0)
        assert (lse.cpu().double() - want).abs().max().item() < 2e-3   # sums of rounded weights: 2^-9, in log2 units


@pytest.mark.gpu
@pytest.mark.parametrize("S", [100, 256])
@pytest.mark.parametrize("fill", [-1e9, float("-inf"), -3e38])
def test_rows_that_attend_nothing_and_large_logits(S, fill):
    """An entry whose every key is masked gives zeros and a statistic of +inf, one with half of its keys masked and logits in the
    hundreds the result of its own keys; the entries beside them are what they are without them."""
    g = torch.Generator().manual_seed(S)
    N, H, D = 5, 2, 32
    q, k, v = (torch.randn(N, H, S, D, generator=g).to(torch.bfloat16) for _ in range(3))
    pair = torch.randn(1, H, S, S, generator=g).to(torch.bfloat16)
    q[3] *= 40
    k[3] *= 10
    row = torch.zeros(N, 1, 1, S).to(torch.bfloat16)
    row[1] = fill
    row[3, ..., S // 2:] = fill
    lse = torch.empty(N, H, S, device=DEV)
    out = _ffi.attn_fwd(q.to(DEV), k.to(DEV), v.to(DEV), biases=[(pair.to(DEV), N), (row.to(DEV), 1)], lse=lse).float().cpu()
    s = q.double() @ k.double().transpose(-1, -2) / D ** 0.5 + pair.double() + row.double()
    ref = torch.softmax(s, -1).nan_to_num() @ v.double()
    ref[1] = 0
    assert (out[1] == 0).all() and (lse[1] == float("inf")).all()
    for n in (0, 2, 3, 4):
        assert ((out[n] - ref[n]).norm() / ref[n].norm()).item() < 3e-3, n


UNEVEN = [(6, 4, 250), (5, 8, 250), (7, 6, 256), (3, 2, 63)]  # batch, divisor that leaves a remainder (or is larger), length


@pytest.mark.parametrize("B,div,S", UNEVEN)
def test_a_batch_that_the_divisor_does_not_divide_goes_elsewhere(B, div, S):
    """Entry n takes bias n / divisor whatever the batch size; the stripe kernel's workgroups walk whole groups of entries."""
    p = params(S=S, lse=0x90000, B=B)
    p.bias_batch_div[0] = div
    plan = _ffi.plan(p)
    assert plan["streaming"] == 0 and plan["workgroups"] == B * p.Hq * -(-S // plan["rows_per_workgroup"])


@pytest.mark.gpu
@pytest.mark.parametrize("B,div,S", UNEVEN)
def test_a_batch_that_the_divisor_does_not_divide(B, div, S):
    g = torch.Generator().manual_seed(B * S)
    H, D, groups = 2, 32, -(-B // div)
    q, k, v = (torch.randn(B, H, S, D, generator=g).to(torch.bfloat16) for _ in range(3))
    pair = torch.randn(groups, H, S, S, generator=g).to(torch.bfloat16)
    lib, dev = _ffi.load_library(), [t.to(DEV) for t in (q, k, v, pair)]
    out = torch.full((B, H, S, D), float("nan"), dtype=torch.bfloat16, device=DEV)
    lse = torch.full((B, H, S), float("nan"), device=DEV)
    p, keep = _ffi._fill_params(lib, *dev[:3], out, H, H, None, 0, 0, 0, None, 0, 0.0, [(dev[3][:1], B)], None, False, 0.0, None)
    p.bias_strides[0][0], p.bias_batch_div[0], p.lse = H * S * S, div, lse.data_ptr()   # (the Python entries refuse such divisors)
    assert lib.fl_attn_fwd(C.byref(p), torch.cuda.current_stream().cuda_stream) == 0, _ffi.last_error()
    s = q.double() @ k.double().transpose(-1, -2) / D ** 0.5 + pair.double()[torch.arange(B) // div]
    ref = torch.softmax(s, -1) @ v.double()
    # weights and results rounded to bf16, as above
    assert ((out.cpu().double() - ref).norm() / ref.norm()).item() < 3e-3
    # every rounded weight is off by at most 2^-8 of its size, and so is their sum: 2^-8 / ln 2 in log2 units (1e-4: the exponential)
    assert (lse.cpu().double() - torch.logsumexp(s, -1) / math.log(2.0)).abs().max().item() < 2.0 ** -8 / math.log(2.0) + 1e-4
    del keep
