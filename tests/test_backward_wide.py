"""Gradients of many heads at head dim 128: workgroups of 256 keys for dK and dV (wide_dkv in csrc/api.hip), against
the unplanned call, whose workgroups have 128 keys and which the other backward tests hold against the oracle."""
import ctypes as C

import pytest
import torch

from flashlight_amd import _ffi
from tests.test_abi import good_params

DEV = "cuda"
NONE, CAUSAL, SLIDING, PREFIX = _ffi.MASK_NONE, _ffi.MASK_CAUSAL, _ffi.MASK_SLIDING, _ffi.MASK_PREFIX_LM


def _plan(B, Hq, Hkv, Lq, Lk, mask, window=70, prefix=40, D=128, **kw):
    """(launches, workgroups per dQ tile, per dK/dV tile, keys per dK/dV workgroup) of the gradients."""
    p = good_params(B=B, Hq=Hq, Hkv=Hkv, L=Lk, D=D)
    p.Lq, p.mask_kind, p.window, p.prefix = Lq, mask, window, prefix
    for name, value in kw.items():
        setattr(p, name, value)
    out = (C.c_int64 * 4)()
    assert _ffi.load_library().fl_attn_bwd_plan(C.byref(p), out) == 0, _ffi.last_error()
    return tuple(out)


def test_which_calls_take_wide_workgroups():
    keys = lambda heads, L, mask, **kw: _plan(1, heads, heads, L, L, mask, **kw)[3]  # noqa: E731
    assert keys(16, 4096, NONE) == 256 and keys(15, 4096, NONE) == 128 and keys(24, 4096, NONE) == 128 and keys(75, 4096, NONE) == 256
    assert keys(129, 2048, NONE) == 256 and keys(43, 6000, NONE) == 128 and keys(49, 6000, NONE) == 256
    for mask in (CAUSAL, PREFIX):  # heads that do not divide by the XCDs: short walks only
        assert keys(128, 2048, mask) == 256 and keys(129, 2048, mask) == 128 and keys(136, 2048, mask) == 256
        assert keys(121, 1000, mask) == 256 and keys(167, 1536, mask) == 256 and keys(81, 1536, mask) == 128 and keys(85, 3000, mask) == 256 and keys(63, 3000, mask) == 128
        assert keys(65, 4096, mask) == 128 and keys(69, 4300, mask) == 256 and keys(63, 4096, mask) == 128
        assert keys(1024, 256, mask) == 256 and keys(1088, 256, mask) == 128 and keys(1089, 256, mask) == 256
    assert keys(129, 2048, SLIDING) == 256 and keys(129, 2048, SLIDING, window=1025) == 128 and keys(121, 1000, SLIDING, window=900) == 256
    assert keys(16, 640, NONE) == 128  # (a tenth of the places of 256 keys would be empty)
    assert keys(16, 4096, NONE, D=64) == 128 and keys(16, 4096, NONE, softcap=30.0) == 128 and keys(16, 4096, NONE, dropout_threshold=99) == 128
    assert keys(16, 4096, _ffi.MASK_DOCUMENT) == 128
    lib = _ffi.load_library()
    out = (C.c_int64 * 4)()
    assert lib.fl_attn_bwd_plan(None, out) == -1 and lib.fl_attn_bwd_plan(C.byref(good_params()), None) == -1
    assert lib.fl_attn_bwd_plan(C.byref(good_params(Hq=3, Hkv=2)), out) == -2


def test_plan_of_the_gradients_follows_the_scratch():
    """Splits are planned where scratch for their sums is asked for, and only there."""
    for call in ((2, 8, 8, 512, 512, CAUSAL), (1, 8, 1, 2048, 2048, CAUSAL), (4, 16, 16, 4096, 4096, CAUSAL), (1, 32, 32, 5876, 5876, NONE)):
        for D in (64, 128):
            launches, dq, dkv, keys = _plan(*call, D=D)
            p = good_params(B=call[0], Hq=call[1], Hkv=call[2], L=call[3], D=D)
            p.mask_kind = call[5]
            assert (_ffi.load_library().fl_attn_bwd_split_bytes(C.byref(p)) > 0) == (dq > 1 or dkv > 1)
            assert launches in (1, 2) and (launches == 1 or (dq, dkv) == (1, 1)) and (launches == 2 or keys == 128)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk,mask", [
    (32, 32, 32, 129, 129, CAUSAL), (32, 16, 16, 256, 256, CAUSAL), (16, 32, 16, 511, 511, CAUSAL), (32, 16, 16, 200, 200, SLIDING),
    (32, 16, 16, 250, 250, PREFIX), (32, 16, 16, 33, 161, NONE), (32, 32, 32, 31, 255, NONE), (16, 32, 16, 300, 400, NONE), (8, 64, 32, 70, 2050, NONE)])
def test_wide_workgroups_give_the_gradients_of_narrow_ones(B, Hq, Hkv, Lq, Lk, mask, dtype):
    g = torch.Generator().manual_seed(Lq + Lk)
    q, k, v, dout = (torch.randn(B, h, n, 128, generator=g).to(dtype).to(DEV) for h, n in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk), (Hq, Lq)))
    kw = dict(mask_kind=mask, window=70, prefix=40)

    assert _plan(B, Hq, Hkv, Lq, Lk, mask) == (2, 1, 1, 256)
    lse = torch.empty(B, Hq, Lq, dtype=torch.float32, device=DEV)
    out = _ffi.attn_fwd(q, k, v, lse=lse, **kw)

    def gradients(split):
        return _ffi.attn_bwd(q, k, v, out, lse, dout, split=split, **kw)

    # The same 16-bit weights and score gradients, added up in another order in fp32 (relative error of a sum of n terms below n * 2^-24 of
    # their magnitudes): results may differ where they round to the other neighbour.  dQ is formed alike.
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for name, a, b in zip(("dq", "dk", "dv"), gradients(True), gradients(False)):
        a, b = a.double(), b.double()
        assert torch.isfinite(a).all(), name
        assert ((a - b).norm(dim=(-2, -1)) < ulp / 4 * b.norm(dim=(-2, -1))).all(), name  # (head by head: one left out or exchanged fails)
        assert ((a - b).abs() <= 2 * ulp * b.abs() + 2e-5 * b.abs().max()).all(), name
