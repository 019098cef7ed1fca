"""The backward of attention with a bias shared by several batch entries (csrc/pairbias_bwd_kernel.h): the Evoformer's
row attention in training, at the edges of its 32-row stripes, wave splits and resident-entry counts, against autograd
through the fp32 oracle."""
import ctypes as C

import pytest
import torch

import flashlight_amd.attention_variants as A
import oracle as O
from flashlight_amd import _ffi, ops
from tests.test_abi import good_params

DEV = "cuda"


def test_which_calls_the_shared_bias_backward_takes():
    lib = _ffi.load_library()
    lib.fl_attn_shared_bias_bwd_bytes.restype = C.c_uint64

    def params(S=256, D=32, H=4, **kw):
        p = good_params(D=D)
        p.B, p.Hq, p.Hkv, p.Lq, p.Lk = 12, H, H, S, S
        p.q_strides[:] = p.k_strides[:] = p.v_strides[:] = p.o_strides[:] = (S * H * D, D, H * D, 1)
        p.bias[0], p.bias_batch_div[0] = 0x60000, 6
        p.bias_strides[0][:] = (H * S * S, S * S, S, 1)
        for n, v in kw.items():
            setattr(p, n, v)
        return p

    takes = lambda p: lib.fl_attn_shared_bias_bwd_bytes(C.byref(p)) > 0  # noqa: E731
    assert takes(params()) and takes(params(S=512, D=64)) and takes(params(S=1))
    assert not takes(params(S=513)) and not takes(params(D=128)) and not takes(params(softcap=3.0))
    assert not takes(params(mask_kind=_ffi.MASK_CAUSAL)) and not takes(params(Hkv=2)) and not takes(params(Lq=128))
    assert not takes(params(H=1 << 15)) and takes(params(H=(1 << 15) - 1))  # rows of [position][head][dim] results: 2^20 elements
    p = params()
    p.bias_strides[0][1] = 0  # one bias for all heads: another sum
    assert not takes(p)
    p = params()
    p.bias[1], p.bias_batch_div[1] = 0x70000, 1
    p.bias_strides[1][:] = (256, 0, 0, 1)
    assert takes(p)
    # a result before the gate goes with a gate, and is named as such in the backward alone
    assert lib.fl_attn_fwd_ungated(C.byref(params()), C.c_void_p(0x90000), None) == -5
    assert lib.fl_attn_fwd_ungated(C.byref(params(gate=0x80000)), C.c_void_p(0x90008), None) == -7
    assert lib.fl_attn_validate(C.byref(params(flags=_ffi.FLAG_UNGATED))) == -5

    class Bwd(C.Structure):  # fl_attn_shared_bias_bwd_params, as far as a refusal looks: its forward's flags come first
        _fields_ = [("fwd", _ffi.FlAttnParams), ("rest", C.c_uint64 * 40)]

    for flags, rc in ((_ffi.FLAG_UNGATED | _ffi.FLAG_SCRATCH, -1), (_ffi.FLAG_F32_RESULT, -5), (4, -5)):   # (-1: no dout)
        assert lib.fl_attn_shared_bias_bwd(C.byref(Bwd(fwd=params(flags=flags))), None) == rc


CASES = [  # B, N, S, H, D
    (1, 3, 32, 2, 32), (2, 5, 64, 3, 32), (1, 9, 100, 4, 64), (2, 17, 129, 2, 32), (1, 4, 256, 4, 64), (1, 40, 256, 8, 32),
    (1, 7, 257, 2, 64), (1, 6, 384, 2, 32), (1, 3, 511, 2, 64), (1, 3, 512, 1, 32), (3, 2, 33, 1, 64), (1, 1, 77, 2, 32)]


@pytest.mark.gpu
@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("shape", CASES)
def test_gradients_against_the_oracle(shape, gate):
    B, N, S, H, D = shape
    g = torch.Generator().manual_seed(sum(shape))
    for dt, mask, f32 in ((torch.bfloat16, False, False), (torch.float16, True, False), (torch.bfloat16, True, True)):
        mk = lambda *s: torch.randn(*s, generator=g).to(dt)  # noqa: E731
        q, k, v, dout = (mk(B, N, S, H, D) for _ in range(4))
        pair = torch.randn(B, 1, H, S, S, generator=g).to(torch.float32 if f32 else dt)
        gl = mk(B, N, S, H, D) if gate else None
        row = None
        if mask:
            row = torch.where(torch.rand(B, N, 1, 1, S, generator=g) < 0.2, float("-inf"), 0.0).to(dt)
            row[..., 0] = 0
        leaves = [t for t in (q, k, v, pair, gl) if t is not None]
        dev = [t.to(DEV).requires_grad_(True) for t in leaves]
        kw = {"gate": dev[4]} if gate else {}
        out = A.attention_reference(dev[0], dev[1], dev[2], ([row.to(DEV)] if mask else []) + [dev[3]], **kw)
        grads = torch.autograd.grad(out, dev, dout.to(DEV))
        ref = [t.float().requires_grad_(True) for t in leaves]
        want = O.attention_evoformer(ref[0], ref[1], ref[2], ([row.float()] if mask else []) + [ref[3]], **({"gate": ref[4]} if gate else {}))
        wgrads = torch.autograd.grad(want, ref, dout.float())
        for name, a, b in zip(("out", "dq", "dk", "dv", "dbias", "dgate"), (out, *grads), (want, *wgrads)):
            rel = ((a.float().cpu() - b).norm() / b.norm()).item()
            assert a.dtype == (torch.float32 if f32 and name == "dbias" else dt) and a.shape == b.shape
            assert rel < (1e-2 if dt == torch.bfloat16 else 3e-3), (shape, gate, mask, f32, name, rel)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(8, 2, 33, 32), (5, 1, 64, 64), (3, 2, 96, 32)])  # B, H, S, D
@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float32])
def test_one_bias_for_the_whole_batch(shape, bias_dtype):
    """A bias with a batch axis of 1 and the divisor left at 1: its gradient is the sum over the batch, and nothing is
    written beside it (the freed slot between tensors of the gradient's size is where the allocator puts it)."""
    B, H, S, D = shape
    g = torch.Generator().manual_seed(sum(shape))
    q, k, v, dout = (torch.randn(B, H, S, D, generator=g).to(torch.bfloat16) for _ in range(4))
    pair = torch.randn(1, H, S, S, generator=g).to(bias_dtype)
    row = torch.randn(B, 1, 1, S, generator=g).to(torch.bfloat16)
    for biases in ([pair], [pair, row], [row, pair]):
        dev = [t.to(DEV).requires_grad_(True) for t in (q, k, v, pair)]
        out = ops.dispatch(*dev[:3], biases=[(dev[3] if b is pair else b.to(DEV), 1) for b in biases])
        around = [torch.full((1, H, S, S), 7.0, dtype=bias_dtype, device=DEV) for _ in range(4 * B)]
        del around[2 * B]
        grads = torch.autograd.grad(out, dev, dout.to(DEV))
        assert all((t == 7.0).all() for t in around)
        ref = [t.float().requires_grad_(True) for t in (q, k, v, pair)]
        s = ref[0] @ ref[1].transpose(-1, -2) / D ** 0.5 + sum(ref[3] if b is pair else b.float() for b in biases)
        want = torch.autograd.grad(torch.softmax(s, -1) @ ref[2], ref, dout.float())
        for name, a, b in zip(("dq", "dk", "dv", "dbias"), grads, want):
            assert a.shape == b.shape
            assert ((a.float().cpu() - b).norm() / b.norm()).item() < 1e-2, (shape, name)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 6, 64, 2, 32), (1, 4, 129, 2, 64)])  # B, N, S, H, D
def test_nearly_closed_gates(shape):
    """fp16, gate logits around -12 under a loss scale: the gated result is mostly below the normal numbers, the gradients
    are not and keep the type's precision.  (Each is a product of a few factors rounded to 11 bits, rms error 2^-11 / sqrt 3
    = 2.8e-4 each; formed from the gated result the gate's gradient is off by 1e-2, dq by 2e-3.)"""
    B, N, S, H, D = shape
    g = torch.Generator().manual_seed(sum(shape))
    q, k, v, dout, gate = (torch.randn(B, N, S, H, D, generator=g) for _ in range(5))
    pair = torch.randn(B, 1, H, S, S, generator=g).half()
    leaves = [q.half(), k.half(), v.half(), pair, (gate - 12.0).half()]
    dout = (1024.0 * dout).half()
    dev = [t.to(DEV).requires_grad_(True) for t in leaves]
    out = A.attention_reference(*dev[:3], [dev[3]], gate=dev[4])
    ref = [t.double().requires_grad_(True) for t in leaves]
    want = O.attention_evoformer(*ref[:3], [ref[3]], gate=ref[4])
    assert ((out.double().cpu() - want).abs() <= 2.0 ** -24 + 2.0 ** -10 * want.abs()).all()  # half a subnormal step, two roundings
    for name, a, b in zip(("dq", "dk", "dv", "dbias", "dgate"), torch.autograd.grad(out, dev, dout.to(DEV)),
                          torch.autograd.grad(want, ref, dout.double())):
        assert ((a.double().cpu() - b).norm() / b.norm()).item() < 1e-3, (shape, name)


@pytest.mark.gpu
def test_output_gradient_with_rows_far_apart():
    """An output gradient whose positions lie 2^20 elements apart, beyond the kernels' offsets, is copied."""
    g = torch.Generator().manual_seed(2)
    q, k, v, gate, dout = (torch.randn(1, 2, 33, 2, 32, generator=g).to(torch.bfloat16).to(DEV).requires_grad_(True) for _ in range(5))
    pair = torch.randn(1, 1, 2, 33, 33, generator=g).to(torch.bfloat16).to(DEV).requires_grad_(True)
    far = torch.empty(33 << 20, dtype=torch.bfloat16, device=DEV).as_strided(dout.shape, (128, 64, 1 << 20, 32, 1))
    far.copy_(dout.detach())
    for kw in ({}, {"gate": gate}):
        leaves = [q, k, v, pair, *kw.values()]
        out = A.attention_reference(q, k, v, [pair], **kw)
        near = torch.autograd.grad(out, leaves, dout.detach(), retain_graph=True)
        assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(out, leaves, far), near))


@pytest.mark.gpu
def test_layouts_partial_gradients_and_repetition():
    """Heads-first operands, gradients of the bias alone or not at all, the same bits twice, and a second derivative that
    is refused instead of missing."""
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(1, 6, 2, 96, 32, generator=g).to(torch.bfloat16).to(DEV).transpose(-2, -3) for _ in range(3))
    pair = torch.randn(1, 1, 2, 96, 96, generator=g).to(torch.bfloat16).to(DEV).requires_grad_(True)
    a, = torch.autograd.grad(A.attention_reference(q, k, v, [pair]).float().square().sum(), [pair])
    q.requires_grad_(True)
    b = torch.autograd.grad(A.attention_reference(q, k, v, [pair]).float().square().sum(), [pair, q])
    c = torch.autograd.grad(A.attention_reference(q, k, v, [pair.detach()]).float().square().sum(), [q])
    assert torch.equal(a, b[0]) and torch.equal(b[1], c[0])
    out = A.attention_reference(q, k, v, [pair])
    dq, = torch.autograd.grad(out.float().sum(), [q], create_graph=True)
    with pytest.raises(RuntimeError, match="not differentiable a second time"):
        dq.float().sum().backward()


def test_scales_that_a_bias_row_cannot_be_divided_by():
    """Bias rows start the products' accumulators, divided by the scale: where that is no ordinary number, another kernel takes the call."""
    lib = _ffi.load_library()
    lib.fl_attn_shared_bias_bwd_bytes.restype = C.c_uint64
    out = (C.c_int64 * 8)()
    for scale, taken in ((1e-39, False), (1e-31, False), (1e-29, True), (0.0, True), (1e29, True), (1e31, False), (3e38, False)):
        for row in (False, True):
            p = good_params(B=12, Hq=4, Hkv=4, L=101, D=32)
            p.scale = scale
            p.bias[0], p.bias_batch_div[0] = 0x60000, 6
            p.bias_strides[0][:] = (4 * 101 * 101, 101 * 101, 101, 1)
            if row:
                p.bias[1], p.bias_batch_div[1] = 0x70000, 1
                p.bias_strides[1][:] = (101, 0, 0, 1)
            assert (lib.fl_attn_shared_bias_bwd_bytes(C.byref(p)) > 0) == (taken or not row), (scale, row)
            if scale:
                assert lib.fl_attn_plan(C.byref(p), out) == 0 and (out[6] == 2) == (taken or not row), (scale, row)


@pytest.mark.gpu
@pytest.mark.parametrize("S", [101, 256])
def test_a_tiny_scale_beside_a_bias_row(S):
    """The products vanish: what is left are the weights of the biases alone, and their gradients."""
    N, H, D = 6, 2, 32
    g = torch.Generator().manual_seed(S)
    q, k, v, dout = (torch.randn(N, H, S, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(4))
    pair = torch.randn(1, H, S, S, generator=g).to(torch.bfloat16).to(DEV)
    row = torch.where(torch.rand(N, 1, 1, S, generator=g) < 0.2, float("-inf"), torch.randn(N, 1, 1, S, generator=g)).to(torch.bfloat16).to(DEV)
    leaves = [t.requires_grad_(True) for t in (q, k, v, pair)]
    out = ops.dispatch(q, k, v, scale=1e-39, biases=[(pair, N), (row, 1)])
    grads = torch.autograd.grad(out, leaves, dout)
    exact = [v.detach().double().requires_grad_(True), pair.detach().double().requires_grad_(True)]
    want = torch.matmul(torch.softmax(exact[1] + row.double(), -1), exact[0])
    wgrads = torch.autograd.grad(want, exact, dout.double())
    for name, a, b in zip(("out", "dv", "dbias"), (out, *grads[2:]), (want, *wgrads)):
        assert ((a.double() - b).norm() / b.norm()).item() < 1e-2, name  # (weights, score gradients and results rounded to bf16)
    assert all((t.abs() < 1e-30).all() for t in grads[:2])
