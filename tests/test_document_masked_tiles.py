"""Masked tiles under documents (TILE_ONE_DOC in csrc/fwd_kernel.h and the ids as bits of the mask's word, there and in csrc/bwd_kernel.h): rows
of one document, whose masked tiles look at no ids, and boundaries at every place of a tile, forward and gradients against attention
in 64 bits."""
import math

import pytest
import torch

from flashlight_amd import _ffi

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(ids, D, H, causal, dtype=torch.bfloat16):
    S, g = ids.numel(), torch.Generator().manual_seed(ids.numel() + D)
    q, k, v, dout = (torch.randn(1, H, S, D, generator=g).to(dtype) for _ in range(4))
    kw = dict(mask_kind=_ffi.MASK_DOCUMENT_CAUSAL if causal else _ffi.MASK_DOCUMENT, doc_ids=ids[None].to(DEV))
    dev = [t.to(DEV) for t in (q, k, v, dout)]
    lse = torch.empty(1, H, S, dtype=torch.float32, device=DEV)
    out = _ffi.attn_fwd(*dev[:3], lse=lse, **kw)
    got = [out] + list(_ffi.attn_bwd(*dev[:3], out, lse, dev[3], **kw))
    ql, kl, vl = (t.double().requires_grad_(True) for t in (q, k, v))
    off = ids[:, None] != ids[None, :]
    if causal:
        off = off | torch.ones(S, S, dtype=torch.bool).triu(1)
    o = torch.softmax((ql @ kl.transpose(-1, -2) / math.sqrt(D)).masked_fill(off, -math.inf), -1) @ vl
    want = [o.detach()] + list(torch.autograd.grad(o, (ql, kl, vl), dout.double()))
    # weights or score gradients, results, and (twice) the forward's result in the row sums, each rounded to the element type: 2^-9 or 2^-12 at most
    eps = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    for name, a, w in zip(("out", "dq", "dk", "dv"), got, want):
        rel = ((a.double().cpu() - w).norm() / w.norm()).item()
        assert rel <= 0.58 * 4 * eps, (S, D, causal, name, rel)


@pytest.mark.parametrize("D,dtype", [(32, torch.bfloat16), (64, torch.bfloat16), (64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("S", [31, 64, 65, 127, 200, 513, 4300])
def test_one_document(S, causal, D, dtype):
    _check(torch.full((S,), -5), D, 2 if S > 4000 else 3, causal, dtype)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_a_boundary_at_every_place_of_a_tile(D, causal):
    for cut in range(61, 132, 1 if D == 64 else 5):
        _check(torch.tensor([7] * cut + [(1 << 40) + 7] * (199 - cut)), D, 2, causal)


@pytest.mark.parametrize("D", [64, 128])
def test_ids_that_alternate_and_come_back(D):
    n = torch.arange(300)
    for ids in (n % 2, n // 70 % 2, (n * 7919) % 5 - 2):  # every tile has several, in runs of every length
        for causal in (False, True):
            _check(ids, D, 2, causal)


@pytest.mark.parametrize("D", [256, 512])
@pytest.mark.parametrize("causal", [False, True])
def test_head_dims_whose_masked_tiles_compare_ids_at_every_score(D, causal):
    S, H = 229, 2
    n = torch.arange(S)
    for ids in (torch.full((S,), -5), n // 70, (n * 7919) % 3, (n >= 101).long() << 40):
        g = torch.Generator().manual_seed(D)
        q, k, v = (torch.randn(1, H, S, d, generator=g).to(torch.bfloat16) for d in (D, D, 128))
        kw = dict(mask_kind=_ffi.MASK_DOCUMENT_CAUSAL if causal else _ffi.MASK_DOCUMENT, doc_ids=ids[None].to(DEV))
        off = ids[:, None] != ids[None, :]
        if causal:
            off = off | torch.ones(S, S, dtype=torch.bool).triu(1)
        for cap in (0.0, 9.0):
            got = _ffi.attn_fwd(q.to(DEV), k.to(DEV), v.to(DEV), softcap=cap, **kw).double().cpu()
            x = q.double() @ k.double().transpose(-1, -2) / math.sqrt(D)
            want = torch.softmax((cap * torch.tanh(x / cap) if cap else x).masked_fill(off, -math.inf), -1) @ v.double()
            # weights and results are each rounded by 2^-8 of themselves at most, 2^-8 / sqrt(3) in the norm (emulated in 64 bits: 2.17e-3 in all)
            assert ((got - want).norm() / want.norm()).item() <= math.sqrt(2 / 3) * 2.0 ** -8, (D, causal, cap)
