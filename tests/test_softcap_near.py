"""Soft-cap of scores that are small beside the cap, which is a polynomial there (NearCap in csrc/fwd_kernel.h), and the way from it to
the exact form where a tile has others, against torch in 64 bits."""
import math

import pytest
import torch

from flashlight_amd import attention_variants as A

pytestmark = pytest.mark.gpu
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,S,heads", [(32, 333, 16), (64, 700, 8), (64, 2100, 3), (128, 450, 16), (128, 1100, 3), (256, 333, 4)])
@pytest.mark.parametrize("alibi,causal", [(False, False), (True, True), (True, False)])
def test_scores_on_both_sides_of_the_range(D, S, heads, dtype, alibi, causal):
    # standard deviation 1.5: at cap 12 the range ends at 3, which some tiles reach and others do not; at 50 none does
    for cap in (12.0, 50.0):
        _check(*_operands(2, heads, S, D, dtype, 7, 1.5), cap, alibi, causal)


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


@pytest.mark.parametrize("cap", [1e-30, 1e-4, 0.05, 300.0, 2e4])
def test_caps_far_from_the_scale(cap):
    q, k, v = _operands(1, 8, 500, 64, torch.bfloat16, 13)
    _check(q, k, v, cap, False, True)


def test_infinite_scores_are_the_cap():
    q, k, v = _operands(1, 8, 640, 64, torch.bfloat16, 17)
    q[..., 0] = q[..., 0].abs() + 0.1
    k[0, :, 200, 0] = math.inf
    k[0, :, 500, 0] = -math.inf
    _check(q, k, v, 5.0, False, False)
