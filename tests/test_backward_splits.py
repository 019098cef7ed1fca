"""Backward tiles cut into several workgroups (fl_attn_bwd_split) against the same call with whole tiles, which the other
backward tests hold against the oracle; which calls are cut, and that the partial sums stay inside the scratch."""
import ctypes as C

import pytest
import torch

from flashlight_amd import _ffi
from tests.test_abi import good_params

DEV = "cuda"


def _split_bytes(B, Hq, Hkv, Lq, Lk, D, mask=_ffi.MASK_NONE, window=0):
    p = good_params(D=D)
    p.B, p.Hq, p.Hkv, p.Lq, p.Lk, p.mask_kind, p.window = B, Hq, Hkv, Lq, Lk, mask, window
    return _ffi.load_library().fl_attn_bwd_split_bytes(C.byref(p))


def test_which_backwards_are_cut():
    assert _split_bytes(4, 16, 16, 4096, 4096, 128, _ffi.MASK_CAUSAL) == 0      # enough tiles
    assert _split_bytes(1, 8, 8, 256, 256, 64) == 0                             # too few steps
    # 3 x 16 heads over 4, 1000 rows: 384 tiles of 16 steps and 96 of 64, half of them attended: a share is 12 steps
    assert _split_bytes(3, 16, 4, 1000, 1000, 64, _ffi.MASK_PREFIX_LM) == 6 * 96 * 128 * 64 * 2 * 4
    # 8 heads over 1, 2048 rows: 128 tiles of 32 steps, 16 of 256
    assert _split_bytes(1, 8, 1, 2048, 2048, 128, _ffi.MASK_CAUSAL) == (2 * 128 + 16 * 16 * 2) * 128 * 128 * 4
    # a window of 100: few steps per tile whatever the length
    assert _split_bytes(1, 2, 2, 8192, 8192, 64, _ffi.MASK_SLIDING, 100) == 0
    assert _ffi.load_library().fl_attn_bwd_split_bytes(None) == 0


CASES = [  # B, Hq, Hkv, Lq, Lk, D, mask, extra
    (3, 16, 4, 1000, 1000, 64, _ffi.MASK_PREFIX_LM, dict(prefix=200)),
    (1, 8, 1, 513, 513, 128, _ffi.MASK_CAUSAL, {}),
    (1, 3, 3, 2047, 2047, 32, _ffi.MASK_NONE, {}),
    (1, 1, 1, 100, 3001, 64, _ffi.MASK_NONE, {}),
    (1, 8, 2, 1025, 77, 128, _ffi.MASK_NONE, dict(softcap=3.0)),
    (2, 4, 1, 1500, 1500, 128, _ffi.MASK_SLIDING, dict(window=700)),
    (1, 4, 4, 1111, 1111, 64, _ffi.MASK_DOCUMENT_CAUSAL, {}),
    (1, 8, 2, 900, 900, 64, _ffi.MASK_CAUSAL, dict(dropout_p=0.25, dropout_seed=11)),
    (1, 5, 5, 1300, 1300, 128, _ffi.MASK_CAUSAL, dict(alibi_heads=5)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_cut_tiles_give_the_gradients_of_whole_tiles(case, dtype, monkeypatch):
    B, Hq, Hkv, Lq, Lk, D, mask, extra = case
    g = torch.Generator().manual_seed(Lq + Lk)
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)  # noqa: E731
    q, k, v, dout = mk(B, Hq, Lq, D), mk(B, Hkv, Lk, D), mk(B, Hkv, Lk, D), mk(B, Hq, Lq, D)
    kw = dict(mask_kind=mask, **extra)
    if mask == _ffi.MASK_DOCUMENT_CAUSAL:
        kw["doc_ids"] = torch.sort(torch.randint(0, 4, (B, Lk), generator=g), dim=1).values.to(DEV)
    lse = torch.empty(B, Hq, Lq, dtype=torch.float32, device=DEV)
    out = _ffi.attn_fwd(q, k, v, lse=lse, **kw)
    lib = _ffi.load_library()
    calls = []

    class Recorded:  # the library with its split entry given a scratch of exactly the asked size, NaN inside and out
        def __getattr__(self, name):
            if name != "fl_attn_bwd_split":
                return getattr(lib, name)

            def entry(params, _scratch, n, stream):
                buf = torch.full((n // 4 + 1024,), float("nan"), device=DEV)
                rc = lib.fl_attn_bwd_split(params, buf.data_ptr(), n, stream)
                calls.append((buf, n))
                return rc
            return entry

    monkeypatch.setattr(_ffi, "load_library", lambda *a: Recorded())
    cut = _ffi.attn_bwd(q, k, v, out, lse, dout, split=True, **kw)
    whole = _ffi.attn_bwd(q, k, v, out, lse, dout, **kw)
    torch.cuda.synchronize()
    (buf, n), = calls
    assert torch.isnan(buf[n // 4:]).all()
    # the same 16-bit weights and score gradients, added up in another order in fp32 (relative error of a sum of n terms
    # below n * 2^-24 of their magnitudes): results may differ where they round to the other neighbour
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for name, a, b in zip(("dq", "dk", "dv"), cut, whole):
        assert torch.isfinite(a).all(), name
        d, ref = (a.double() - b.double()), b.double()
        assert (d.norm() / ref.norm()).item() < ulp / 4, name
        assert (d.abs() <= 2 * ulp * ref.abs() + 2e-5 * ref.abs().max()).all(), name


LONG_WALKS = [  # cut though no tile is longer than one and a half shares; more splits than the share asks for; documents' shares
    (44, 16, 2, 512, 100, 128, _ffi.MASK_NONE, {}),
    (90, 8, 1, 2000, 100, 32, _ffi.MASK_NONE, {}),
    (6, 8, 2, 1900, 1900, 128, _ffi.MASK_DOCUMENT_CAUSAL, {}),
]


def test_which_long_walks_are_cut():
    sums = lambda splits, tiles, D: splits * tiles * 128 * D * 2 * 4  # noqa: E731
    assert [_split_bytes(*c[:7]) for c in LONG_WALKS] == [sums(2, 88, 128), sums(4, 90, 32), sums(2, 180, 128)]
    assert _split_bytes(12, 8, 1, 3000, 3000, 64) == sums(2, 288, 64)
    assert _split_bytes(16, 8, 1, 3000, 3000, 64) == 0   # a walk of 0.75 shares
    assert _split_bytes(10, 16, 4, 2000, 2000, 64) == 0  # one launch, whole tiles


@pytest.mark.gpu
@pytest.mark.parametrize("case", LONG_WALKS)
def test_long_walks_give_the_gradients_of_whole_tiles(case, monkeypatch):
    test_cut_tiles_give_the_gradients_of_whole_tiles(case, torch.bfloat16, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("mask", [_ffi.MASK_NONE, _ffi.MASK_CAUSAL, _ffi.MASK_DOCUMENT_CAUSAL])
def test_both_roles_in_one_launch_beyond_a_round(mask, D):
    """528 tiles of keys: the same bits as the two halves, which have 256 and 272."""
    g = torch.Generator().manual_seed(D)
    q, k, v, dout = (torch.randn(33, h, 70, D, generator=g).to(torch.bfloat16).to(DEV) for h in (32, 16, 16, 32))
    ids = torch.sort(torch.randint(0, 3, (33, 70), generator=g), dim=1).values.to(DEV)

    def gradients(part):
        kw = dict(mask_kind=mask, **(dict(doc_ids=ids[part]) if mask == _ffi.MASK_DOCUMENT_CAUSAL else {}))
        lse = torch.empty(*q[part].shape[:3], dtype=torch.float32, device=DEV)
        out = _ffi.attn_fwd(q[part], k[part], v[part], lse=lse, **kw)
        return _ffi.attn_bwd(q[part], k[part], v[part], out, lse, dout[part], split=True, **kw)

    for whole, a, b in zip(gradients(slice(None)), gradients(slice(0, 16)), gradients(slice(16, 33))):
        assert torch.equal(whole, torch.cat([a, b]))


@pytest.mark.gpu
@pytest.mark.parametrize("run", [1, 3, 64])
@pytest.mark.parametrize("shape", [(1, 1, 1, 2000, 64), (1, 2, 1, 2000, 128), (1, 1, 1, 3000, 128)])
def test_splits_that_find_no_live_tile(shape, run):
    """Documents so short that a tile of keys has fewer live tiles of queries than it has splits (four and more)."""
    B, Hq, Hkv, S, D = shape
    assert _split_bytes(B, Hq, Hkv, S, S, D, _ffi.MASK_DOCUMENT_CAUSAL) >= 4 * Hkv * -(-S // 128) * 128 * D * 2 * 4
    g = torch.Generator().manual_seed(S + run)
    q, k, v, dout = (torch.randn(B, h, S, D, generator=g).to(torch.bfloat16).to(DEV) for h in (Hq, Hkv, Hkv, Hq))
    kw = dict(mask_kind=_ffi.MASK_DOCUMENT_CAUSAL, doc_ids=(torch.arange(S) // run * 5 - 9)[None].to(DEV))
    lse = torch.empty(B, Hq, S, dtype=torch.float32, device=DEV)
    out = _ffi.attn_fwd(q, k, v, lse=lse, **kw)
    cut = _ffi.attn_bwd(q, k, v, out, lse, dout, split=True, **kw)
    for a, b in zip(cut, _ffi.attn_bwd(q, k, v, out, lse, dout, **kw)):
        # the same 16-bit weights and score gradients, added up in another order: as above
        assert torch.isfinite(a).all() and ((a.double() - b.double()).abs() <= 2.0 ** -7 * b.double().abs() + 2e-5 * v.abs().max()).all()
    if run == 1:  # one key per query: the weights are 1
        want = dout.double().view(B, Hkv, Hq // Hkv, S, D).sum(2)
        assert ((cut[2].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -9 * dout.abs().max()).all()
