"""Forward calls of few workgroups: 64-row workgroups and groups of waves that share the rows and take a part of the key tiles each
(plan_few in csrc/api.hip), against the same rows in a call of many workgroups, whose waves walk all tiles in order."""
import ctypes as C

import pytest
import torch

from flashlight_amd import _ffi
from tests.test_abi import good_params

DEV = "cuda"
NONE, CAUSAL, SLIDING, PREFIX, DOC, DOC_CAUSAL = (_ffi.MASK_NONE, _ffi.MASK_CAUSAL, _ffi.MASK_SLIDING, _ffi.MASK_PREFIX_LM,
                                                  _ffi.MASK_DOCUMENT, _ffi.MASK_DOCUMENT_CAUSAL)


def _shape(B, H, S, D, mask, **kw):
    """(rows per workgroup, groups of waves) the library plans."""
    p = good_params(B=B, Hq=H, Hkv=H, L=S, D=D)
    p.mask_kind, p.window, p.prefix = mask, 300, 100
    if mask in (DOC, DOC_CAUSAL):
        p.doc_ids, p.workspace, p.workspace_bytes = 0x50000, 0x80000, 1 << 30
    for n, v in kw.items():
        setattr(p, n, v)
    out = (C.c_int64 * 8)()
    assert _ffi.load_library().fl_attn_plan(C.byref(p), out) == 0, _ffi.last_error()
    return out[0], out[7]


def test_which_calls_take_groups():
    for mask in (CAUSAL, PREFIX):
        assert _shape(2, 8, 2048, 64, mask) == (64, 2)                   # one workgroup of 128 rows per compute unit
        assert _shape(1, 8, 2048, 64, mask) == (64, 4)                   # half of that, long walks
        assert _shape(1, 16, 3000, 64, mask) == (64, 2)                  # up to two per compute unit, few heads
        assert _shape(8, 16, 1100, 64, mask) == (128, 1)                 # many heads
        assert _shape(4, 16, 4096, 64, mask) == (128, 1)
        assert _shape(1, 8, 4096, 128, mask) == (64, 2) and _shape(1, 16, 3000, 128, mask) == (128, 2)
        assert _shape(4, 16, 512, 128, mask) == (128, 1) and _shape(2, 4, 700, 32, mask) == (128, 1)
    assert _shape(1, 8, 4096, 64, NONE) == (128, 2) and _shape(1, 16, 4096, 64, NONE) == (128, 1)
    assert _shape(1, 4, 4096, 64, NONE) == (64, 4) and _shape(1, 4, 4096, 128, SLIDING, window=1000) == (64, 2)
    assert _shape(1, 8, 4096, 128, SLIDING) == (128, 2) and _shape(2, 16, 2100, 128, SLIDING) == (128, 1)
    # the shape of the lists does not depend on the heads
    assert _shape(2, 16, 1000, 64, DOC) == (128, 2) and _shape(4, 16, 1000, 64, DOC) == (128, 1)
    assert _shape(1, 16, 5000, 64, DOC_CAUSAL) == (128, 2) and _shape(1, 32, 5000, 64, DOC_CAUSAL) == (128, 1)
    assert _shape(2, 8, 1000, 128, CAUSAL, alibi_heads=8, softcap=3.0) == (64, 2)
    assert _shape(2, 8, 1000, 128, CAUSAL, dropout_threshold=1000) == (128, 1)
    assert _shape(1, 1, 4096, 64, CAUSAL) == (128, 1) and _shape(6, 16, 250, 64, CAUSAL) == (128, 1)    # one head; walks of few tiles
    assert _shape(6, 16, 512, 64, NONE)[1] == 1 and _shape(6, 16, 128, 64, DOC)[1] == 1 and _shape(6, 16, 200, 64, DOC)[1] == 2


SIZES = {  # (batch, heads, rows, keys): parts of one tile and none, odd parts, ragged last tiles, four groups
    CAUSAL: [(2, 16, 257, 257), (2, 18, 384, 384), (2, 16, 385, 385), (5, 8, 513, 513), (6, 2, 1025, 1025), (2, 5, 1983, 1983),
             (6, 8, 40, 390), (6, 8, 500, 390)],
    PREFIX: [(2, 18, 385, 385), (2, 16, 449, 449), (3, 4, 1100, 1100)],
    SLIDING: [(8, 6, 385, 385), (3, 10, 700, 700), (2, 10, 900, 900), (2, 4, 1500, 1500)],
    NONE: [(12, 8, 129, 641), (3, 10, 700, 700), (2, 8, 200, 1025), (3, 3, 1100, 1100), (4, 16, 300, 1500)],
    DOC: [(2, 6, 193, 193), (2, 6, 255, 255), (2, 6, 1000, 1000)],
    DOC_CAUSAL: [(2, 6, 193, 193), (1, 6, 300, 300), (2, 6, 777, 777)],
}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("mask,mods", [(m, False) for m in SIZES] + [(CAUSAL, True), (NONE, True)])
def test_groups_give_the_rows_of_a_large_call(mask, mods, D, dtype):
    for B, H, Lq, Lk in SIZES[mask]:
        g = torch.Generator().manual_seed(Lq + Lk + D)
        mk = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)  # noqa: E731
        q, k, v = mk(B, H, Lq, D), mk(B, H // (2 if H % 2 == 0 else 1), Lk, D), mk(B, H // (2 if H % 2 == 0 else 1), Lk, D)
        kw = dict(mask_kind=mask)
        if mask == SLIDING:
            kw["window"] = 260 if Lk < 1000 else 1100
        if mask == PREFIX:
            kw["prefix"] = 100
        if mask in (DOC, DOC_CAUSAL):
            ids = torch.randint(0, 5, (B, Lk), generator=g)
            kw["doc_ids"] = (ids if Lk == 1000 else ids.sort(dim=1).values).to(DEV)
        if mods:
            kw.update(alibi_heads=H, softcap=8.0)
        times = -(-1100 // (B * H * -(-Lq // 128)))
        many = {n: t.repeat(times, 1) if n == "doc_ids" else t for n, t in kw.items()}
        r = lambda t: t.repeat(times, 1, 1, 1)  # noqa: E731
        lse, lse_many = (torch.empty(n, H, Lq, dtype=torch.float32, device=DEV) for n in (B, B * times))
        out = _ffi.attn_fwd(q, k, v, lse=lse, **kw)
        ref = _ffi.attn_fwd(r(q), r(k), r(v), lse=lse_many, **many)[:B].double()
        mean_abs = _ffi.attn_fwd(r(q), r(k), r(v.abs()), **many)[:B].double()  # sum of weight * |value|
        # Weights are rounded to 16 bits relative to another reference (u of their size; fp16 weights far below it are subnormal, together
        # less than 2^-15 of the row's sum), numerator and row sum alike; the result is rounded once more: both sides may be off by
        # u (mean_abs + |o|) + u |o|.  Row statistics: u of the sum.  (a quarter more with a soft-cap, whose exponential is approximate)
        u = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) * (1.25 if mods else 1.0)
        bound = 2 * (u * (mean_abs + 2 * ref.abs()) + 2.0 ** -15 * v.abs().max().item())
        case = f"B={B} H={H} Lq={Lq} Lk={Lk}"
        assert torch.isfinite(out).all(), case
        assert ((out.double() - ref).abs() <= bound).all(), case
        assert ((lse - lse_many[:B]).abs() <= 2 * 1.4427 * u + 1e-4).all(), case


@pytest.mark.gpu
def test_groups_keep_infinities_and_empty_parts_apart():
    """A part all of whose weights vanish beside the others' maximum, one that attends nothing, and a NaN that stays in its rows."""
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(1, 8, 1100, 64, generator=g).to(torch.bfloat16).to(DEV) for _ in range(3))
    k[:, :, 700:] *= 300  # logits of thousands in the last part only
    q[:, :, 500, 0] = float("nan")
    ref = _ffi.attn_fwd(*(t.repeat(16, 1, 1, 1) for t in (q, k, v)), mask_kind=CAUSAL)[:1]
    out = _ffi.attn_fwd(q, k, v, mask_kind=CAUSAL)
    assert torch.equal(out.isnan(), ref.isnan()) and out[:, :, 500].isnan().all() and out.isnan().sum().item() == 8 * 64
    assert (out.nan_to_num().float() - ref.nan_to_num().float()).abs().max().item() <= 2.0 ** -5  # (values of 1 to 4: two roundings)


def test_which_calls_take_64_row_workgroups():
    assert _shape(16, 16, 700, 64, CAUSAL) == (64, 1) and _shape(16, 16, 1024, 64, CAUSAL) == (128, 1)
    assert _shape(15, 8, 151, 64, CAUSAL) == (128, 1) and _shape(30, 16, 151, 64, CAUSAL) == (64, 1)
    assert _shape(16, 16, 128, 64, CAUSAL) == (128, 1) and _shape(16, 16, 700, 128, CAUSAL) == (128, 1)
    assert _shape(16, 16, 700, 64, PREFIX, prefix=350) == (64, 1) and _shape(16, 16, 700, 64, PREFIX, prefix=351) == (128, 1)
    assert _shape(4, 16, 4096, 64, SLIDING, window=895) == (64, 1) and _shape(4, 16, 4096, 64, SLIDING, window=896) == (128, 1)
    assert _shape(4, 16, 4096, 64, NONE) == (128, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("mask,kw", [(CAUSAL, {}), (PREFIX, dict(prefix=60)), (SLIDING, dict(window=70)), (SLIDING, dict(window=300))])
@pytest.mark.parametrize("S", [129, 191, 192, 193, 500])
def test_64_row_workgroups_against_fp64(mask, kw, S):
    g = torch.Generator().manual_seed(S)
    q, k, v = (torch.randn(8, 66, S, 64, generator=g).to(torch.bfloat16).to(DEV) for _ in range(3))
    out = _ffi.attn_fwd(q, k, v, mask_kind=mask, **kw)[7].double()
    i = torch.arange(S, device=DEV)
    d = i[:, None] - i[None, :]
    live = (d >= 0) & (d <= kw.get("window", S)) | (i[None, :] < kw.get("prefix", 0))
    w = torch.softmax((torch.matmul(q[7].double(), k[7].double().transpose(1, 2).contiguous()) / 8).masked_fill(~live, -torch.inf), -1)
    ref, mean_abs = torch.matmul(w, v[7].double()), torch.matmul(w, v[7].double().abs())
    # weights rounded to u = 2^-8 of their size, numerator and row sum alike, and the result once more
    assert ((out - ref).abs() <= 2.0 ** -8 * (mean_abs + 2 * ref.abs()) + 1e-5).all()


ATTENDED = [  # mask, options, (batch, heads, length, head dim), (rows per workgroup, groups of waves)
    (CAUSAL, {}, (2, 8, 2048, 64), (64, 2)), (CAUSAL, {}, (1, 8, 2047, 64), (64, 4)), (CAUSAL, {}, (1, 16, 3000, 128), (128, 2)),
    (CAUSAL, {}, (2, 18, 385, 64), (64, 2)), (CAUSAL, {}, (1, 8, 1025, 128), (64, 2)),
    (PREFIX, dict(prefix=333), (2, 8, 1100, 64), (64, 2)), (PREFIX, dict(prefix=1000), (1, 8, 1500, 64), (64, 4)),
    (PREFIX, dict(prefix=70), (1, 8, 900, 128), (64, 2)),
    (SLIDING, dict(window=300), (1, 8, 4000, 128), (128, 2)), (SLIDING, dict(window=1000), (1, 4, 2500, 128), (64, 2)),
    (SLIDING, dict(window=1300), (1, 4, 2500, 64), (64, 4)),
    (NONE, {}, (1, 8, 2100, 128), (128, 2)), (NONE, {}, (1, 4, 3001, 64), (64, 4)), (NONE, {}, (1, 8, 4096, 64), (128, 2)),
    (DOC, {}, (2, 16, 1000, 64), (128, 2)), (DOC, {}, (1, 16, 1500, 128), (128, 2)), (DOC_CAUSAL, {}, (1, 16, 5000, 64), (128, 2)),
    (DOC_CAUSAL, {}, (2, 8, 777, 128), (128, 2)),
]


def _attended(mask, kw, S, g):
    """Which key each row attends, and the options of the call."""
    i = torch.arange(S, device=DEV)
    d = i[:, None] - i[None, :]
    live = torch.ones(S, S, dtype=torch.bool, device=DEV) if mask in (NONE, DOC) else d >= 0
    call = dict(kw, mask_kind=mask)
    if mask == SLIDING:
        live &= d <= kw["window"]
    if mask == PREFIX:
        live |= (i < kw["prefix"])[None, :]
    if mask in (DOC, DOC_CAUSAL):
        ids = torch.randint(0, 6, (S,), generator=g).sort().values.to(DEV)
        ids[S // 3] = 5  # (a document that comes back)
        live &= ids[:, None] == ids[None, :]
        call["doc_ids"] = ids[None]
    return live, call


@pytest.mark.gpu
@pytest.mark.parametrize("mask,kw,shape,plan", ATTENDED)
def test_which_keys_the_groups_attend(mask, kw, shape, plan):
    """Read off the results, as the dump of attended pairs runs without groups: equal logits, and values that are the unit vectors,
    a block of D keys per (batch, head).  Row q then holds 1 / n at each of the n keys it attends, and 0 at every other."""
    B, H, S, D = shape
    assert _shape(B, H, S, D, mask, **kw) == plan
    g = torch.Generator().manual_seed(S)
    live, call = _attended(mask, kw, S, g)
    q = torch.zeros(B, H, S, D, dtype=torch.bfloat16, device=DEV)
    k = torch.randn(B, H, S, D, generator=g).to(torch.bfloat16).to(DEV)
    found = torch.empty(S, -(-S // D) * D, device=DEV)
    for first in range(0, -(-S // D), B * H):
        v = torch.zeros(B * H, S, D, dtype=torch.bfloat16, device=DEV)
        for bh in range(B * H):
            at = (first + bh) * D
            n = max(0, min(D, S - at))
            v[bh, at:at + n] = torch.eye(D, dtype=torch.bfloat16, device=DEV)[:n]
        out = _ffi.attn_fwd(q, k, v.view(B, H, S, D), **call).float().view(B * H, S, D)
        for bh in range(min(B * H, -(-S // D) - first)):
            found[:, (first + bh) * D:(first + bh + 1) * D] = out[bh]
    want = live / live.sum(1, keepdim=True)
    assert torch.equal(found[:, :S] != 0, live)
    # equal logits: every weight is 1 and the sums are exact, or off together; one rounding of the result
    assert ((found[:, :S] - want).abs() <= 2.0 ** -8 * want).all()


@pytest.mark.gpu
@pytest.mark.parametrize("mask,kw,shape,plan", [c for c in ATTENDED if c[2][2] <= 2100])
def test_groups_against_fp64(mask, kw, shape, plan):
    B, H, S, D = shape
    g = torch.Generator().manual_seed(S + 1)
    q, k, v = (torch.randn(B, H, S, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(3))
    live, call = _attended(mask, kw, S, g)
    out = _ffi.attn_fwd(q, k, v, **call)[-1].double()
    w = torch.softmax((torch.matmul(q[-1].double(), k[-1].double().transpose(1, 2).contiguous()) / D ** 0.5).masked_fill(~live, -torch.inf), -1)
    ref, mean_abs = torch.matmul(w, v[-1].double()), torch.matmul(w, v[-1].double().abs())
    # weights rounded to u = 2^-8 of their size, numerator and row sum alike, and the result once more
    assert ((out - ref).abs() <= 2.0 ** -8 * (mean_abs + 2 * ref.abs()) + 1e-5).all()
