"""The gradients' lists of live tiles under a document mask (csrc/bwd_kernel.h): ragged ends, ids that come back far apart, more tiles
than one list holds, grouped heads and cut tiles, against attention within each document in fp32."""
import pytest
import torch

from flashlight_amd import _ffi

DEV = "cuda"


def _ids(kind, S, g):
    """Runs of random length; `again`: the first document comes back at every tenth run and at the end."""
    ids, n = [], 0
    while sum(len(x) for x in ids) < S:
        run = int(torch.randint(1, max(2, min(400, S // 2)), (1,), generator=g))
        ids.append(torch.full((run,), 0 if kind == "again" and n % 10 == 0 else n * 7 - 3, dtype=torch.int64))
        n += 1
    ids = torch.cat(ids)[:S]
    if kind == "again":
        ids[-1] = ids[0]
    return ids


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["runs", "again"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("S,D,H,G", [(33, 64, 1, 2), (200, 128, 2, 2), (777, 64, 2, 4), (1500, 32, 1, 1), (67000, 64, 1, 1), (35000, 128, 1, 2)])
def test_live_tiles(S, D, H, G, causal, kind):
    g = torch.Generator().manual_seed(S)
    B = 1 if S > 10000 else 2
    mk = lambda h: torch.randn(B, h, S, D, generator=g).to(torch.bfloat16)  # noqa: E731
    q, k, v, dout = mk(H * G), mk(H), mk(H), mk(H * G)
    ids = torch.stack([_ids(kind, S, g) for _ in range(B)])
    kw = dict(mask_kind=_ffi.MASK_DOCUMENT_CAUSAL if causal else _ffi.MASK_DOCUMENT, doc_ids=ids.to(DEV))
    dev = [t.to(DEV) for t in (q, k, v, dout)]
    lse = torch.empty(B, H * G, S, dtype=torch.float32, device=DEV)
    out = _ffi.attn_fwd(*dev[:3], lse=lse, **kw)
    got = [_ffi.attn_bwd(*dev[:3], out, lse, dev[3], split=split, **kw) for split in (False, True)]
    want = [torch.zeros(t.shape) for t in (q, k, v)]
    for b in range(B):
        for doc in ids[b].unique():
            at = (ids[b] == doc).nonzero().flatten()
            n = len(at)
            if n > 3000:  # (the document that keeps coming back in the long case: its first and last positions are enough)
                continue
            ql, kl, vl = (t[b][:, at].float().requires_grad_(True) for t in (q, k, v))
            s = ql @ kl.repeat_interleave(G, 0).transpose(-1, -2) / D ** 0.5
            if causal:
                s = s.masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), float("-inf"))
            o = torch.softmax(s, -1) @ vl.repeat_interleave(G, 0)
            for w, x in zip(want, torch.autograd.grad(o, (ql, kl, vl), dout[b][:, at].float())):
                w[b][:, at] = x
    for grads in got:
        for name, a, w in zip(("dq", "dk", "dv"), grads, want):
            a = a.float().cpu()
            seen = (w != 0).any(-1)
            assert seen.float().mean() > 0.8
            rel = ((a - w)[seen].norm() / w[seen].norm()).item()
            assert rel < 1e-2, (S, D, causal, kind, name, rel)
