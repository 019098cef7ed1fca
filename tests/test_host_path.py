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
