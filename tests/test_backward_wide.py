"""Gradients of many heads at head dim 128: workgroups of 256 keys for dK and dV (wide_dkv in csrc/api.hip), against the same heads in a call of
few, whose workgroups have 128 keys and which the other backward tests hold against the oracle."""
import pytest
import torch

from flashlight_amd import _ffi

DEV = "cuda"
NONE, CAUSAL, SLIDING, PREFIX = _ffi.MASK_NONE, _ffi.MASK_CAUSAL, _ffi.MASK_SLIDING, _ffi.MASK_PREFIX_LM


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk,mask", [
    (32, 32, 32, 129, 129, CAUSAL), (32, 16, 16, 256, 256, CAUSAL), (16, 32, 16, 511, 511, CAUSAL), (32, 16, 16, 200, 200, SLIDING),
    (32, 16, 16, 250, 250, PREFIX), (32, 16, 16, 33, 161, NONE), (32, 32, 32, 31, 255, NONE), (16, 32, 16, 300, 400, NONE), (8, 64, 32, 70, 2050, NONE)])
def test_wide_workgroups_give_the_gradients_of_narrow_ones(B, Hq, Hkv, Lq, Lk, mask, dtype):
    g = torch.Generator().manual_seed(Lq + Lk)
    q, k, v, dout = (torch.randn(B, h, n, 128, generator=g).to(dtype).to(DEV) for h, n in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk), (Hq, Lq)))
    kw = dict(mask_kind=mask, window=70, prefix=40)

    lse = torch.empty(B, Hq, Lq, dtype=torch.float32, device=DEV)
    out = _ffi.attn_fwd(q, k, v, lse=lse, **kw)

    def gradients(part, split):
        q_, k_, v_, o_, l_, d_ = (t[part].contiguous() for t in (q, k, v, out, lse, dout))
        return _ffi.attn_bwd(q_, k_, v_, o_, l_, d_, split=split, **kw)

    # The same 16-bit weights and score gradients, added up in another order in fp32 (relative error of a sum of n terms below n * 2^-24 of
    # their magnitudes): results may differ where they round to the other neighbour.  dQ is formed alike.
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for name, a, b in zip(("dq", "dk", "dv"), gradients(slice(0, B), True), gradients(slice(B - 1, B), False)):
        a, b = a[B - 1:].double(), b.double()
        assert torch.isfinite(a).all(), name
        assert ((a - b).norm() / b.norm()).item() < ulp / 4, name
        assert ((a - b).abs() <= 2 * ulp * b.abs() + 2e-5 * b.abs().max()).all(), name
