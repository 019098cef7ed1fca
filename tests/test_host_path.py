"""The native host path of the front ends (csrc/host.cpp): what it takes, and that it behaves as the Python path does."""
import ctypes as C

import pytest
import torch

from flashlight_amd import _ffi, ops

DEV = "cuda"


def _operands(*shape, dtype=torch.bfloat16, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(*shape, generator=g).to(dtype).to(DEV) for _ in range(3)]


@pytest.mark.gpu
def test_other_threads_run_while_a_call_is_launched():
    """The library's entries replaced by CPython's own question whether this thread holds the interpreter: it returns 1,
    which the host path reads as a refusal, or 0, a launch."""
    lib = _ffi.load_library()
    address = {f: C.cast(getattr(lib, f), C.c_void_p).value for f in _ffi._HOST_ENTRIES}
    asked = C.cast(C.pythonapi.PyGILState_Check, C.c_void_p).value
    q, k, v = _operands(1, 2, 64, 64)
    pair = torch.zeros(1, 2, 64, 64, dtype=torch.bfloat16, device=DEV)
    args = (None, 0, 0, 0, None, 0, 0.0)
    try:
        _ffi._host.bind(*(asked if f in ("fl_attn_fwd", "fl_attn_bwd_split", "fl_attn_shared_bias_bwd") else a for f, a in address.items()))
        assert _ffi._host.forward(q, k, v, *args, (), None, False, 0.0, False) is not None
        q.requires_grad_(True)
        for biases in ((), ((pair, 1),)):
            out = _ffi._host.forward(q, k, v, *args, biases, None, False, 0.0, False)
            assert out is not None
            torch.autograd.grad(out, [q], torch.zeros_like(out))
    finally:
        _ffi._host.bind(*address.values())
    q.requires_grad_(False)
    assert torch.isfinite(ops.dispatch(q, k, v)).all()


@pytest.mark.gpu
def test_the_first_call_goes_the_way_of_the_others(monkeypatch):
    """The library is loaded by the first call, which takes the native path like every later one (a differentiable gated
    call rounds its result once there, twice in the Python path's composition)."""
    q, k, v = _operands(4, 2, 64, 32)
    gate, = _operands(4, 2, 64, 32, seed=1)[:1]
    pair = torch.randn(1, 2, 64, 64, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).to(DEV)
    q.requires_grad_(True)
    call = lambda: ops.dispatch(q, k, v, biases=[(pair, 4)], gate=gate)  # noqa: E731
    later = call()
    monkeypatch.setattr(_ffi, "_lib", None)
    monkeypatch.setattr(_ffi, "_host", None)
    assert torch.equal(call(), later)


class _PythonPath:
    """The native module with a `forward` that takes no call."""

    def __init__(self, host):
        self.key_chunks = host.key_chunks

    def forward(self, *args):
        return None


def _both(monkeypatch, run):
    """run() by the native path and by the Python path."""
    native = run()
    with monkeypatch.context() as m:
        m.setattr(_ffi, "_host", _PythonPath(_ffi._host))
        return native, run()


def _same(a, b, exact=True):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.dtype == y.dtype
        if exact:
            assert torch.equal(x, y)
        else:  # (another order of sums, and one rounding less under a gate: each is within 3.2e-3 or 4e-4 of the exact one)
            assert ((x.float() - y.float()).norm() / y.float().norm()).item() < (6e-3 if x.dtype == torch.bfloat16 else 1e-3)


def _layouts(B, H, S, D, dtype):
    """q, k, v of [B, H, S, D] in layouts that callers have: as they lie addressable by the kernels or not."""
    g = torch.Generator().manual_seed(S)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)  # noqa: E731
    yield "contiguous", [r(B, H, S, D) for _ in range(3)]
    yield "projection", [t.transpose(1, 2) for t in r(B, S, 3, H, D).unbind(2)]
    yield "slice of a longer buffer", [t[:, :, 3:3 + S] for t in r(3, B, H, S + 9, D)]
    yield "one head for all", [r(B, H, S, D), r(B, 1, S, D).expand(B, H, S, D), r(B, 1, S, D).expand(B, H, S, D)]
    yield "off by one element", [r(B, H, S, D + 8)[..., 1:D + 1] for _ in range(3)]
    yield "rows of 65 elements", [r(B, H, S, D + 1)[..., :D] for _ in range(3)]
    yield "dims first", [r(B, H, D, S).transpose(2, 3) for _ in range(3)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(2, 4, 77, 64), (1, 2, 300, 128), (3, 2, 128, 32)])
def test_layouts_of_operands_and_gradients(shape, dtype, monkeypatch):
    _ffi.load_library()
    B, H, S, D = shape
    g = torch.Generator().manual_seed(9)
    flat = torch.randn(B, H, S, D, generator=g).to(dtype).to(DEV)
    douts = [flat, flat.transpose(1, 2).contiguous().transpose(1, 2), flat[:, :, :1].expand_as(flat), flat.transpose(2, 3).contiguous().transpose(2, 3),
             torch.randn(B, H, S, D + 3, generator=g).to(dtype).to(DEV)[..., 1:D + 1]]
    for name, ops3 in _layouts(*shape, dtype):
        for kw in ({}, dict(mask_kind=_ffi.MASK_CAUSAL), dict(softcap=4.0, alibi_heads=H, mask_kind=_ffi.MASK_SLIDING, window=30)):
            _same(*_both(monkeypatch, lambda: [ops.dispatch(*ops3, **kw)]))
            leaves = [t.detach().requires_grad_(True) for t in ops3]
            for dout in douts:
                _same(*_both(monkeypatch, lambda: torch.autograd.grad(ops.dispatch(*leaves, **kw), leaves, dout)))


@pytest.mark.gpu
@pytest.mark.parametrize("gate", [False, True])
def test_shared_bias_calls(gate, monkeypatch):
    _ffi.load_library()
    q, k, v = _operands(6, 2, 70, 32)
    extra = _operands(6, 2, 70, 32, seed=1)
    g = torch.Generator().manual_seed(2)
    pair = torch.randn(2, 2, 70, 70, generator=g).to(torch.bfloat16).to(DEV)
    row = torch.randn(6, 1, 1, 70, generator=g).to(torch.bfloat16).to(DEV)
    leaves = [t.requires_grad_(True) for t in (q, k, v, pair, extra[0])][:5 if gate else 4]
    gates = dict(gate=leaves[4]) if gate else {}
    for biases in ([(pair, 3)], [(pair, 3), (row, 1)], [(row, 1), (pair, 3)], [(pair[:1], 1)], [(pair[:1], 6), (row[:1], 1)]):
        for seq_major in (False, True):
            def run():
                out = ops.dispatch(q, k, v, biases=biases, seq_major_out=seq_major, **gates)
                return [out.detach(), *torch.autograd.grad(out, leaves, extra[1])]
            _same(*_both(monkeypatch, run), exact=False)


@pytest.mark.gpu
def test_autograd_around_the_native_node(monkeypatch):
    """What goes with a node of torch's autograd goes with this one: hooks on saved tensors, anomaly mode, the check for
    in-place changes, one backward per graph, Parameters, partial gradients, calls made on another stream."""
    _ffi.load_library()
    q, k, v = _operands(2, 2, 96, 64)
    dout = torch.randn_like(q)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    pair = torch.zeros(1, 2, 96, 96, dtype=torch.bfloat16, device=DEV)
    for kw in (dict(mask_kind=_ffi.MASK_CAUSAL), dict(biases=[(pair, 2)])):
        want = torch.autograd.grad(ops.dispatch(q, k, v, **kw), leaves, dout)
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.to(DEV)):
            out = ops.dispatch(q, k, v, **kw)
        _same(torch.autograd.grad(out, leaves, dout, retain_graph=True), want)
        assert len(packed) >= 5
        _same(torch.autograd.grad(out, leaves, dout), want)
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(out, leaves, dout)
        with torch.autograd.detect_anomaly(check_nan=True):
            _same(torch.autograd.grad(ops.dispatch(q, k, v, **kw), leaves, dout), want)
        _same(torch.autograd.grad(ops.dispatch(q.detach(), k.detach(), v, **kw), [v], dout), want[2:])
        params = [torch.nn.Parameter(t.detach().clone()) for t in leaves]
        _same(torch.autograd.grad(ops.dispatch(*params, **kw), params, dout), want, exact="biases" not in kw)

        def changed():
            x = q.detach().clone().requires_grad_(True)
            y = x * 1.0
            out = ops.dispatch(y, k, v, **kw)
            with torch.no_grad():
                y.add_(1.0)
            with pytest.raises(RuntimeError, match="modified by an inplace operation"):
                torch.autograd.grad(out, [x], dout)
            return []
        _both(monkeypatch, changed)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            out = ops.dispatch(q, k, v, **kw)
        torch.cuda.current_stream().wait_stream(side)
        got = torch.autograd.grad(out, leaves, dout)
        torch.cuda.synchronize()
        _same(got, want)
