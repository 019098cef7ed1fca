"""The element masks of the forward and the gradients, one bit of a word per score: which scores count, exactly, at every offset of an interval's ends
within a block.  With queries of zero every attended weight is 1/n, so unit vectors as values (or as output gradients, or as keys) make the
forward (dV, dQ) the pattern of the mask itself; what each predicate attends is the reference's (attention_variants/sliding_window.py:14-44,
attention_variants/prefix_lm.py)."""
import ctypes as C

import pytest
import torch

from flashlight_amd import _ffi
from tests.test_abi import good_params

DEV = "cuda"
CAUSAL, SLIDING, PREFIX = _ffi.MASK_CAUSAL, _ffi.MASK_SLIDING, _ffi.MASK_PREFIX_LM
SIZES = [(CAUSAL, 0), *((SLIDING, w) for w in (*range(0, 34), 63, 64, 65, 126)), *((PREFIX, n) for n in (*range(2, 34), 63, 64, 65, 126))]


@pytest.mark.gpu
@pytest.mark.parametrize("B,H", [(1, 4), (8, 8)])  # few heads: from 65 keys on, at head dim 128, the forward's few-rows kernel
@pytest.mark.parametrize("D,length", [(64, 64), (64, 61), (128, 128), (128, 127), (128, 97), (128, 33), (128, 31), (128, 1)])
def test_every_end_of_an_interval(D, length, B, H):
    g = torch.Generator().manual_seed(length)
    p = good_params(B=B, Hq=H, Hkv=H, L=length, D=D)
    p.mask_kind = CAUSAL
    assert _ffi.load_library().fl_attn_rows_plan(C.byref(p), C.byref(C.c_uint64())) == (H == 4 and length > 64)
    random = lambda: (torch.rand(B, H, length, D, generator=g) + 0.5).to(torch.bfloat16).to(DEV)
    unit = torch.eye(D)[:length].to(torch.bfloat16).expand(B, H, length, D).contiguous().to(DEV)
    q, some = torch.zeros_like(unit), random()
    i, j = torch.arange(length)[:, None], torch.arange(length)[None, :]
    for mask, size in SIZES:
        kw = dict(mask_kind=mask, window=size, prefix=size)
        attended = (i >= j) & (i - j <= size) if mask == SLIDING else (i >= j) | ((j < size) if mask == PREFIX else False)
        expected = attended.double() / attended.sum(-1, keepdim=True)
        lse = torch.empty(B, H, length, dtype=torch.float32, device=DEV)
        out = _ffi.attn_fwd(q, unit, unit, lse=lse, **kw)
        weights = out[..., :length].double().cpu()
        assert torch.equal(weights != 0, attended.expand_as(weights)), (mask, size)
        # 1/n formed in fp32 from weights of 1 and rounded to bf16
        assert ((weights - expected).abs() <= 2.0 ** -8 * expected).all(), (mask, size)
        for split in (False, True):
            dv = _ffi.attn_bwd(q, unit, unit, out, lse, unit, split=split, **kw)[2][..., :length].double().cpu()
            assert torch.equal(dv != 0, attended.T.expand_as(dv)), (mask, size, split)
            # a weight rounded to bf16, times 1, and rounded again
            assert ((dv - expected.T).abs() <= 2.0 ** -7 * expected.T).all(), (mask, size, split)
            o = _ffi.attn_fwd(q, unit, some, lse=lse, **kw)
            dq = _ffi.attn_bwd(q, unit, some, o, lse, some, split=split, **kw)[0][..., :length].double().cpu()
            assert (dq[~attended.expand_as(dq)] == 0).all(), (mask, size, split)
            # The score gradient of each pair: sums of D products in fp32 (relative error of the sum of their magnitudes below D 2^-24, for dP and
            # for Delta), rounded to bf16, scaled and rounded again
            vd, od = some.double().cpu(), o.double().cpu()
            dp, delta = torch.matmul(vd, vd.transpose(-1, -2).contiguous()), (vd * od).sum(-1, keepdim=True)
            want = D ** -0.5 * expected * (dp - delta)
            slack = D ** -0.5 * expected * D * 2.0 ** -24 * (dp.abs() + delta.abs())
            assert ((dq - want).abs() <= 2.0 ** -7 * want.abs() + slack).all(), (mask, size, split)
