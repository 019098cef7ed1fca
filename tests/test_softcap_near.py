"""Soft-cap of scores that are small beside the cap, which is a polynomial there (NearCap in csrc/fwd_kernel.h) in calls of some length
(near_cap_pays in csrc/api.hip), and the way from it to the exact form where a tile has others, against torch in 64 bits."""
import math
import subprocess

import numpy as np
import pytest
import torch

from flashlight_amd import _ffi
from flashlight_amd import attention_variants as A
from flashlight_amd import build as B

gpu = pytest.mark.gpu
DEV = "cuda"


def _reference(q, k, v, cap, alibi, causal):
    q, k, v = (t.double().cpu() for t in (q, k, v))
    x = q @ k.transpose(-1, -2) / math.sqrt(q.shape[-1])
    s = cap * torch.tanh(x / cap)
    L, S = s.shape[-2:]
    rel = torch.arange(S)[None, :] - torch.arange(L)[:, None]
    if alibi:
        H = q.shape[1]
        s = s + torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)], dtype=torch.float64)[:, None, None] * rel
    if causal:
        s = s.masked_fill(rel > 0, -math.inf)
    return torch.softmax(s, -1) @ v


def _call(q, k, v, cap, alibi, causal):
    if alibi:
        return A.attention_pytorch_alibi(q, k, v, score_mod=A.generate_alibi_bias_pytorch(q.shape[1]), is_causal=causal, softcap=cap)
    return A.attention_softcapped(q, k, v, score_mod=A.generate_tanh_softcap(cap), is_causal=causal)


def _check(q, k, v, cap, alibi, causal):
    out = _call(q, k, v, cap, alibi, causal).double().cpu()
    ref = _reference(q, k, v, cap, alibi, causal)
    assert torch.isfinite(out).all()
    # weights and results are each rounded to the element type (2^-9 or 2^-12 at most, 0.58 of it in the norm), their products summed in fp32
    eps = 2.0 ** -9 if q.dtype == torch.bfloat16 else 2.0 ** -12
    assert ((out - ref).norm() / ref.norm()).item() <= 2.0 * eps
    return out, ref


def _operands(B, H, S, D, dtype, seed, amplitude=1.0):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, H, S, D, generator=g) for _ in range(3))
    return (q * amplitude).to(dtype).to(DEV), k.to(dtype).to(DEV), v.to(dtype).to(DEV)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,S,heads", [(32, 333, 16), (64, 700, 8), (64, 2100, 3), (128, 450, 16), (128, 1100, 3), (256, 333, 4)])
@pytest.mark.parametrize("alibi,causal", [(False, False), (True, True), (True, False)])
def test_scores_on_both_sides_of_the_range(D, S, heads, dtype, alibi, causal):
    # standard deviation 1.5: at cap 12 the range ends at 3, which every tile reaches; at 50 none does
    for cap in (12.0, 50.0):
        _check(*_operands(2, heads, S, D, dtype, 7, 1.5), cap, alibi, causal)


@gpu
@pytest.mark.parametrize("D,alibi", [(64, False), (64, True), (128, False), (128, True)])
@pytest.mark.parametrize("far", [2.5, -2.5])
def test_one_score_far_out_in_any_place_of_a_tile(D, alibi, far):
    # head h: one query meets one key at far * cap, in tile 1 + h % 5 at place 7 h of it; every register and half of a wave has one
    H, S, cap = 64, 64 * 6, 30.0
    q, k, v = _operands(1, H, S, D, torch.bfloat16, 11)
    q[..., 0] = 0.0
    k[..., 0] = 0.0
    for h in range(H):
        key = 64 * (1 + h % 5) + 7 * h % 64
        q[0, h, 64 + 5 * h % 320, 0] = 16.0
        k[0, h, key, 0] = far * cap * math.sqrt(D) / 16.0
    out, ref = _check(q, k, v, cap, alibi, False)
    for h in range(H):  # the row itself (the polynomial at 2.5 is four times the cap)
        row = 64 + 5 * h % 320
        assert ((out - ref)[0, h, row].norm() / ref[0, h, row].norm()).item() <= 2.0 ** -6


@gpu
@pytest.mark.parametrize("cap", [1e-30, 1e-4, 0.05, 300.0, 2e4])
def test_caps_far_from_the_scale(cap):
    q, k, v = _operands(1, 8, 500, 64, torch.bfloat16, 13)
    _check(q, k, v, cap, False, True)


@gpu
def test_infinite_scores_are_the_cap():
    q, k, v = _operands(1, 8, 640, 64, torch.bfloat16, 17)
    q[..., 0] = q[..., 0].abs() + 0.1
    k[0, :, 200, 0] = math.inf
    k[0, :, 500, 0] = -math.inf
    _check(q, k, v, 5.0, False, False)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,B,S,heads", [(32, 2, 1030, 8), (64, 4, 708, 16), (128, 4, 700, 16), (256, 1, 1100, 4)])
@pytest.mark.parametrize("alibi,causal", [(False, False), (True, True)])
def test_scores_on_both_sides_of_the_range_in_calls_with_the_polynomial(D, B, S, heads, dtype, alibi, causal):
    # standard deviation 1.5: the range ends at 4 and 4.5 of it, which some tiles of a wave's reach and others do not, and at 8, which none does
    q, k, v = _operands(B, heads, S, D, dtype, 7, 1.5)
    x = (q[:1].float() @ k[:1].float().transpose(-1, -2)).abs().cpu() / math.sqrt(D)
    tiles = torch.nn.functional.pad(x, (0, -S % 64, 0, -S % 32)).unflatten(-1, (-1, 64)).unflatten(-3, (-1, 32)).amax((-1, -3))
    for cap in (24.0, 27.0, 50.0):
        outside = tiles > cap / 4
        assert not outside.any() if cap == 50.0 else (outside.any(-1) & ~outside.all(-1)).any()
        _check(q, k, v, cap, alibi, causal)


@gpu
@pytest.mark.parametrize("D,alibi", [(64, False), (64, True), (128, False), (128, True)])
@pytest.mark.parametrize("far", [2.5, -2.5, 0.3])
def test_one_score_far_out_in_any_place_of_a_tile_of_the_polynomial(D, alibi, far):
    # as above, in a call that is long enough for it: head h has its pair in tile 1 + h % 10 at place 7 h of it
    H, S, cap = 64, 64 * 11, 30.0
    q, k, v = _operands(1, H, S, D, torch.bfloat16, 11)
    q[..., 0] = 0.0
    k[..., 0] = 0.0
    for h in range(H):
        q[0, h, 64 + 5 * h % 640, 0] = 16.0
        k[0, h, 64 * (1 + h % 10) + 7 * h % 64, 0] = far * cap * math.sqrt(D) / 16.0
    out, ref = _check(q, k, v, cap, alibi, False)
    for h in range(H):
        row = 64 + 5 * h % 640
        assert ((out - ref)[0, h, row].norm() / ref[0, h, row].norm()).item() <= 2.0 ** -6


def _near_caps(pairs, tmp_path):
    """NearCap::of(scale, cap) of the header, for each pair: (a, b, last, per_last, least, least_well)"""
    try:
        cc = B.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    source, program = tmp_path / "near.hip", tmp_path / "near"
    source.write_text('''#include <cstdio>
#include <cstdlib>
#include "fwd_kernel.h"
int main(int n, char** v) {
  for (int i = 1; i + 1 < n; i += 2) {
    const fl::NearCap c = fl::NearCap::of(std::strtof(v[i], nullptr), std::strtof(v[i + 1], nullptr));
    std::printf("%a %a %a %a %u %u\\n", c.a, c.b, c.last, c.per_last, c.least, c.least_well);
  }
}
''')
    subprocess.run([cc, "-O1", f"--offload-arch={B.ARCH}", "-std=c++17", "--cuda-host-only", f"-I{B.INCLUDE}", f"-I{B.CSRC}", "-x", "hip",
                    str(source), "-o", str(program)], check=True, stderr=subprocess.DEVNULL)
    out = subprocess.run([str(program), *(repr(float(x)) for pair in pairs for x in pair)], check=True, capture_output=True, text=True).stdout
    rows = [line.split() for line in out.splitlines()]
    return [tuple(np.float32(float.fromhex(x)) for x in row[:4]) + tuple(np.uint32(int(x)) for x in row[4:]) for row in rows]


def test_the_polynomial_against_64_bits(tmp_path):
    fma = lambda a, b, c: (a.astype(np.float64) * b + c).astype(np.float32)  # noqa: E731  (rounded twice; the products are exact)
    pairs = [(64 ** -0.5, 50.0), (128 ** -0.5, 50.0), (64 ** -0.5, 30.0), (128 ** -0.5, 12.0), (1.0, 2.0), (0.3, 2e4), (1e-5, 1e-4), (0.125, 0.05)]
    rng = np.random.default_rng(1)
    for (scale, cap), (a, b, last, per_last, least, least_well) in zip(pairs, _near_caps(pairs, tmp_path)):
        scale, cap = float(np.float32(scale)), float(np.float32(cap))
        x = (np.concatenate([rng.uniform(-0.25, 0.25, 400000), rng.normal(0, 0.01, 100000)]) * cap / scale).astype(np.float32)
        u = fma(x, x, a)
        got = (x * fma(u, u, b)).astype(np.float32).astype(np.float64) * last  # (the last product is exact in the kernel's multiply-add)
        want = cap * np.tanh(x.astype(np.float64) * scale / cap) / math.log(2)
        # truncation 4.2e-7 of the score, 1.05e-7 of the cap at the range's end, and three roundings of 2^-24 of terms of up to 1.3 and 1.1 times the score
        assert np.abs(got - want).max() <= 1.4e-7 * cap / math.log(2)
        assert (np.abs(got - want) <= 6.5e-7 * np.abs(want)).all()
        assert abs(per_last * last - 1) < 1e-6
        # which scores it takes: up to a quarter of the cap (five sixths of that), beyond, infinite, not a number
        bits = lambda y: fma(np.float32([y * cap / scale]), np.float32(y * cap / scale), a).view(np.uint32)[0]  # noqa: E731
        for limit, edge in ((least, 0.25), (least_well, 0.25 * 5 / 6)):
            assert all(bits(y) >= limit for y in (0.0, 0.1, -0.1, edge * 0.9999, -edge * 0.9999))
            assert all(bits(y) < limit for y in (edge * 1.0001, -edge * 1.0001, 0.6, 3.0, -1e9, np.inf)) and np.float32(np.nan).view(np.uint32) < limit


def test_scales_that_the_polynomial_leaves_alone(tmp_path):
    # (last = 0: the kernel with the exponential)
    for c in _near_caps([(0.125, 1e-30), (0.125, 1e30), (0.0, 50.0), (-0.125, 50.0), (1e30, 50.0), (1e-30, 1e-30), (math.nan, 50.0), (0.125, math.inf)], tmp_path):
        assert c[2] == 0


@gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_whose_scores_are_all_at_one_place_of_the_range(D, dtype):
    # Scores of a row: one place of the range, -1.2 to 1.2 quarters of the cap, and a few units around it; the cap is so large that a deviation of
    # 1e-6 of it would show in the weights of tiles that take the polynomial beside those that do not: a wave's first tile, here with values that make
    # its weights count, and all beyond the range.  (One head, which groups of waves do not share: a walk of 1024 keys and more takes that kernel.)
    S, cap, rows = 1056, 2e4, 32
    places = torch.tensor([0.02, -0.1, 0.15, 0.2, -0.2, 0.207, 0.212, 0.24, -0.245, 0.26, 0.3, -0.3])
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(1, 1, S, D, generator=g) for _ in range(3))
    v[:, :, :64] *= 16.0
    at = places.repeat_interleave(rows).repeat(S // (rows * len(places)) + 1)[:S]
    # (fp16 holds no more than 65504, so the place is the product of two numbers)
    k[..., 0] = 64.0
    q[..., 0] = at * cap * math.sqrt(D) / 64.0
    q[..., 1:] *= 0.5
    q, k, v = (t.to(dtype) for t in (q, k, v))
    want = _reference(q, k, v, cap, False, False)
    got = A.attention_softcapped(q.to(DEV), k.to(DEV), v.to(DEV), score_mod=A.generate_tanh_softcap(cap), is_causal=False).double().cpu()
    # either form's scores are off by 1.4e-7 or 1.6e-7 of the cap and by the roundings of numbers of up to 0.3 cap log2(e) (2^-24 each, of the products' sum,
    # the score and its addend), which is the relative deviation of a weight; weights and results are rounded besides
    eps = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    bound = (1.4e-7 + 1.6e-7) * cap + 3 * 2.0 ** -24 * 0.3 * cap * 1.45 + 2.0 * eps
    for r in range(0, S, rows):
        rel = ((got - want)[:, :, r:r + rows].norm() / want[:, :, r:r + rows].norm()).item()
        assert rel <= bound, (r, at[r].item(), rel, bound)


def _operands_with_far_pairs(far, kind, S, D, heads, dtype, seed, cap):
    """Scores well inside the range but for some queries' with one key, far from the first that they attend, which are +-far times the cap."""
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(1, heads, S, D, generator=g) for _ in range(3))
    q[..., 0] = 0.0
    k[..., 0] = 0.0
    for h in range(heads):
        rows = [S - 1, S - 2] + [(519 + 520 * (j % 2) if kind == "documents" else S - 1 - 50 * j) - (7 * h + 11 * j) % 48 for j in range(8)]
        keys = [S - 1, S - 2] + [row - (53 * (j + 1) * (h + 2)) % (300 if kind == "documents" else 600) for j, row in enumerate(rows[2:])]
        for i, (row, key) in enumerate(zip(rows, keys)):
            q[0, h, row, 0] = 16.0
            k[0, h, key, 0] = (-far if i % 2 else far) * cap * math.sqrt(D) / 16.0
    return [t.to(dtype) for t in (q, k, v)]


def _attended(kind, S):
    rel = torch.arange(S)[None, :] - torch.arange(S)[:, None]
    ids = torch.arange(S) // 520
    return {"none": torch.ones(S, S, dtype=torch.bool), "causal": rel <= 0, "window": (rel <= 0) & (rel >= -900),
            "documents": (rel <= 0) & (ids[:, None] == ids[None, :])}[kind], ids


@gpu
@pytest.mark.parametrize("far", [0.235, 0.27, 2.5])  # past five sixths of the range (inside it: nothing is formed again), past its end
@pytest.mark.parametrize("kind,D,dtype,alibi,bias,S,heads", [
    ("none", 32, torch.bfloat16, True, False, 1093, 3), ("causal", 32, torch.float16, False, False, 1093, 3),
    ("causal", 256, torch.bfloat16, True, False, 1093, 3), ("none", 512, torch.bfloat16, True, False, 1093, 3),
    # (head dims 64 and 128: one head, or so many keys that each of several groups of waves walks 1024)
    ("causal", 64, torch.float16, True, False, 1093, 1), ("causal", 128, torch.bfloat16, True, False, 1093, 1),
    ("causal", 64, torch.bfloat16, True, False, 4200, 2), ("none", 128, torch.float16, False, False, 2150, 2),
    ("window", 64, torch.bfloat16, True, False, 1093, 1), ("window", 128, torch.float16, False, False, 1093, 1),
    ("documents", 64, torch.bfloat16, True, False, 1093, 1), ("documents", 128, torch.float16, True, False, 1093, 1),
    # (bias operands: the exponential throughout)
    ("none", 64, torch.bfloat16, False, True, 1096, 3), ("none", 128, torch.float16, True, True, 1096, 3),
    ("causal", 64, torch.float16, False, True, 1093, 3), ("none", 32, torch.bfloat16, False, True, 1096, 3)])
def test_waves_that_leave_the_polynomial_on_the_way(kind, D, dtype, alibi, bias, S, heads, far):
    cap = 60.0
    q, k, v = _operands_with_far_pairs(far, kind, S, D, heads, dtype, 31, cap)
    mask, ids = _attended(kind, S)
    x = q.double() @ k.double().transpose(-1, -2) / math.sqrt(D) / cap
    outside = (x.abs() > 0.25 * (5 / 6 if far < 0.25 else 1)) & mask
    # some blocks of a wave's 32 rows and a tile's 64 keys have such scores, after the first tile that the rows attend; one is the last tile
    blocks = lambda t: torch.nn.functional.pad(t.float(), (0, -S % 64, 0, -S % 32)).unflatten(-1, (-1, 64)).unflatten(-3, (-1, 32)).amax((-1, -3)) > 0  # noqa: E731
    far_blocks, first = blocks(outside), blocks(mask).float().argmax(-1)
    start_inside = ~far_blocks.gather(-1, first[None, None, :, None].expand(1, heads, -1, 1))[..., 0]
    assert (far_blocks.any(-1) & start_inside).sum() >= 4 and (far_blocks[..., -1] & start_inside).any()
    scores = cap * torch.tanh(x)
    kw = dict(softcap=cap, mask_kind={"none": _ffi.MASK_NONE, "causal": _ffi.MASK_CAUSAL, "window": _ffi.MASK_SLIDING, "documents": _ffi.MASK_DOCUMENT_CAUSAL}[kind])
    if kind == "window":
        kw["window"] = 900
    if kind == "documents":
        kw["doc_ids"] = ids[None].to(DEV)
    if alibi:
        kw["alibi_heads"] = heads
        rel = (torch.arange(S)[None, :] - torch.arange(S)[:, None]).double()
        scores = scores + torch.tensor([2.0 ** (-8.0 * (h + 1) / heads) for h in range(heads)], dtype=torch.float64)[:, None, None] * rel
    if bias:  # a dense operand, a row of keys, and the gate
        g = torch.Generator().manual_seed(5)
        dense, row, gate = torch.randn(1, heads, S, S, generator=g).to(dtype), torch.randn(1, 1, 1, S, generator=g).to(dtype), torch.randn(1, heads, S, D, generator=g).to(dtype)
        kw.update(biases=[(dense.to(DEV), 1), (row.to(DEV), 1)], gate=gate.to(DEV))
        scores = scores + dense.double() + row.double()
    got = _ffi.attn_fwd(q.to(DEV), k.to(DEV), v.to(DEV), **kw).double().cpu()
    want = torch.softmax(scores.masked_fill(~mask, -math.inf), -1) @ v.double()
    if bias:
        want = want * torch.sigmoid(gate.double())
    # weights and results (and the gated result) rounded to the element type
    eps = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    assert torch.isfinite(got).all() and ((got - want).norm() / want.norm()).item() <= 2.0 * eps
    for h, r in torch.nonzero(outside.any(-1)[0]):
        # (one row, of few values where one weight is not nearly all)
        assert ((got - want)[0, h, r].norm() / want[0, h, r].norm()).item() <= 4.0 * eps, (h, r)
