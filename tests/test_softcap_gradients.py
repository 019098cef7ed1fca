"""Gradients under the soft-cap at head dims 64 and 128 (run_ordered in csrc/bwd_kernel.h: masked positions are taken out of finished
weights), and under ALiBi alone, which has kernels of its own there, against torch in 64 bits."""
import math

import pytest
import torch

from flashlight_amd import attention_variants as A

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _reference(q, k, v, dout, cap, alibi, causal):
    q, k, v = (t.detach().double().cpu().requires_grad_(True) for t in (q, k, v))
    s = q @ k.transpose(-1, -2) / math.sqrt(q.shape[-1])
    if cap:
        s = cap * torch.tanh(s / cap)
    L, S = s.shape[-2:]
    rel = torch.arange(S)[None, :] - torch.arange(L)[:, None]
    if alibi:
        H = q.shape[1]
        s = s + torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)], dtype=torch.float64)[:, None, None] * rel
    if causal:
        s = s.masked_fill(rel > 0, -math.inf)
    return torch.autograd.grad(torch.softmax(s, -1) @ v, (q, k, v), dout.double().cpu())


def _gradients(q, k, v, dout, cap, alibi, causal):
    q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
    if alibi:
        out = A.attention_pytorch_alibi(q, k, v, score_mod=A.generate_alibi_bias_pytorch(q.shape[1]), is_causal=causal, softcap=cap or None)
    else:
        out = A.attention_softcapped(q, k, v, score_mod=A.generate_tanh_softcap(cap), is_causal=causal)
    return torch.autograd.grad(out, (q, k, v), dout.view(out.shape))


def _check(q, k, v, dout, cap, alibi, causal):
    got = [g.double().cpu() for g in _gradients(q, k, v, dout, cap, alibi, causal)]
    ref = _reference(q, k, v, dout, cap, alibi, causal)
    # the weights or score gradients, the results, and the forward's result in the row sums are each rounded to the element type (2^-9 or 2^-12 at
    # most, 0.58 of it in the norm); the row sums' share, which a score gradient is a difference with, counts twice
    eps = 2.0 ** -9 if q.dtype == torch.bfloat16 else 2.0 ** -12
    for g, r in zip(got, ref):
        assert torch.isfinite(g).all()
        assert ((g - r).norm() / r.norm()).item() <= 0.58 * (1 + 1 + 2) * eps
    return got, ref


def _operands(B, H, S, D, dtype, seed, amplitude=1.0):
    g = torch.Generator().manual_seed(seed)
    q, k, v, dout = (torch.randn(B, H, S, D, generator=g) for _ in range(4))
    return [(q * amplitude).to(dtype).to(DEV)] + [t.to(dtype).to(DEV) for t in (k, v, dout)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,S,heads", [(64, 97, 2), (64, 700, 8), (64, 2100, 3), (128, 33, 2), (128, 450, 16), (128, 1100, 3)])
@pytest.mark.parametrize("alibi,causal", [(False, False), (True, True)])
def test_lengths_that_end_inside_a_tile(D, S, heads, dtype, alibi, causal):
    for cap in (2.0, 12.0, 50.0):
        _check(*_operands(2, heads, S, D, dtype, 7, 1.5), cap, alibi, causal)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("far", [2.5, -2.5])
def test_one_score_far_out_in_any_place_of_a_tile(D, far):
    # head h: one query meets one key at far * cap, in tile 1 + h % 5 at place 7 h of it; every register and half of a wave has one.  The pair's
    # weight stays below a tenth: a row that one key has to itself has no gradient but its rounding
    H, S, cap = 64, 64 * 6, 4.0
    q, k, v, dout = _operands(1, H, S, D, torch.bfloat16, 11, 0.15)
    q[..., 0] = 0.0
    k[..., 0] = 0.0
    rows, keys = [64 + 5 * h % 320 for h in range(H)], [64 * (1 + h % 5) + 7 * h % 64 for h in range(H)]
    for h in range(H):
        q[0, h, rows[h], 0] = 16.0
        k[0, h, keys[h], 0] = far * cap * math.sqrt(D) / 16.0
    got, ref = _check(q, k, v, dout, cap, False, False)
    for h in range(H):  # the derivative there is 0.03.  With score gradients and the forward's result rounded, in 64 bits otherwise, the rows below differ by 0.003 at most
        for g, r, at in ((got[0], ref[0], rows[h]), (got[1], ref[1], keys[h])):
            assert ((g - r)[0, h, at].norm() / r[0, h, at].norm()).item() <= 2.0 ** -6


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("cap", [0.05, 300.0, 2e4, 0.0])
def test_caps_far_from_the_scale(D, cap):
    # (0: ALiBi alone)
    _check(*_operands(1, 8, 500, D, torch.bfloat16, 13), cap, cap == 0.0, True)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,heads", [(31, 2), (700, 8), (1100, 3)])
def test_alibi_alone(D, dtype, S, heads):
    for causal in (False, True):
        _check(*_operands(2, heads, S, D, dtype, 19), 0.0, True, causal)


@pytest.mark.parametrize("D", [64, 128])
def test_masked_scores_far_above_the_others(D):
    # keys past the diagonal whose weights against the rows' statistics are infinite
    S, cap = 300, 200.0
    q, k, v, dout = (t.float().cpu() for t in _operands(1, 8, S, D, torch.bfloat16, 23))
    k = k + torch.arange(S)[:, None] / S * 9 * q.mean(2, keepdim=True).sign()
    q = q + k.mean(2, keepdim=True).sign()
    q, k, v, dout = (t.to(torch.bfloat16).to(DEV) for t in (q, k, v, dout))
    got, ref = _gradients(q, k, v, dout, cap, False, True), _reference(q, k, v, dout, cap, False, True)
    # what rounding weights, score gradients, the forward's result and the gradients leaves, in 64 bits otherwise (the keys have a large common
    # part, which the score gradients of a row cancel but for their rounding)
    q, k, v, dout = (t.double().cpu() for t in (q, k, v, dout))
    th = torch.tanh(q @ k.transpose(-1, -2) / math.sqrt(D) / cap)
    past = torch.ones(S, S, dtype=torch.bool).triu(1)
    scores = (cap * th).masked_fill(past, -math.inf)
    assert ((cap * th - torch.logsumexp(scores, -1, keepdim=True))[..., past] > 128 * math.log(2)).any()
    rounded = lambda t: t.to(torch.bfloat16).double()
    P = torch.softmax(scores, -1)
    ds = rounded(P * (dout @ v.transpose(-1, -2) - (dout * rounded(P @ v)).sum(-1, keepdim=True)) * (1 - th * th))
    model = (ds @ k / math.sqrt(D), ds.transpose(-1, -2) @ q / math.sqrt(D), rounded(P).transpose(-1, -2) @ dout)
    for g, m, r in zip(got, model, ref):
        assert ((g.double().cpu() - r).norm() / r.norm()).item() <= 2 * ((rounded(m) - r).norm() / r.norm()).item()
