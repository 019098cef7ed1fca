"""The shared-bias kernels' walks over batch entries: the order of workgroups with neighbours on one XCD, and rows touched ahead of
their transfers in the gradients of calls whose operands are larger than the caches (csrc/tile_operands.h, pairbias_bwd_kernel.h).  Neither
changes a sum, so a part of the entries alone, which takes neither, has the same bits."""
import math

import pytest
import torch

from flashlight_amd import attention_variants as A
from flashlight_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gradients(q, k, v, pair, gate, dout):
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v, gate, pair)]
    out = A.attention_reference(*leaves[:3], [leaves[4]], gate=leaves[3])
    return [out.detach(), *torch.autograd.grad(out, leaves, dout)]


def _pair_gradient(q, k, v, pair, dout, head):
    """In 64 bits, for one head: q, k, v, dout [N, S, H, D] (dout behind the gate), pair [H, S, S] of the entries' group."""
    q, k, v, dout = (t[:, :, head].double().contiguous() for t in (q, k, v, dout))
    p = torch.softmax(q @ k.transpose(1, 2).contiguous() / math.sqrt(q.shape[-1]) + pair[head].double(), -1)
    dp = dout @ v.transpose(1, 2).contiguous()
    return (p * (dp - (p * dp).sum(-1, keepdim=True))).sum(0)


def _check_pair_gradient(got, q, k, v, pair, dout):
    # weights' statistics, row sums and the result rounded to bf16 at 2^-9 at most, of entries that do not add up coherently
    for b in range(pair.shape[0]):
        for head in range(pair.shape[2]):
            want = _pair_gradient(q[b], k[b], v[b], pair[b, 0], dout[b], head)
            assert ((got[b, 0, head].double() - want).norm() / want.norm()).item() <= 1e-2, (b, head)


@pytest.mark.parametrize("N,S,H,D", [(161, 259, 8, 32), (97, 450, 8, 32), (101, 256, 7, 64), (95, 391, 5, 64)])  # more than 80 MB of q, k, v, dout
def test_entries_of_a_large_call_are_those_of_a_small_one(N, S, H, D):
    assert N * S * H * D * 8 > 80 << 20
    g = torch.Generator(device=DEV).manual_seed(N)
    q, k, v, gate, dout = (torch.randn(1, N, S, H, D, generator=g, device=DEV).bfloat16() for _ in range(5))
    pair = torch.randn(1, 1, H, S, S, generator=g, device=DEV).bfloat16()
    large = _gradients(q, k, v, pair, gate, dout)
    for first in (0, N // 2, N - 3):
        part = [t[:, first:first + 3].contiguous() for t in (q, k, v, gate, dout)]
        small = _gradients(part[0], part[1], part[2], pair, part[3], part[4])
        for name, a, b in zip(("out", "dq", "dk", "dv", "dgate"), large, small):
            assert torch.equal(a[:, first:first + 3], b), (name, first)
    _check_pair_gradient(large[5], q, k, v, pair, (dout.double() * torch.sigmoid(gate.double())))


@pytest.mark.parametrize("B,N,S,H,D", [(2, 110, 300, 5, 32), (3, 41, 200, 7, 32), (2, 47, 333, 3, 64), (1, 30, 384, 9, 32)])
def test_groups_of_entries_and_units_that_do_not_divide_by_eight(B, N, S, H, D):
    # (the first also touches rows ahead; the forward's chunks are of 5 entries and more)
    assert B * N * S * H * D * 8 > 24 << 20
    g = torch.Generator(device=DEV).manual_seed(N)
    q, k, v, gate, dout = (torch.randn(B, N, S, H, D, generator=g, device=DEV).bfloat16() for _ in range(5))
    pair = torch.randn(B, 1, H, S, S, generator=g, device=DEV).bfloat16()
    large = _gradients(q, k, v, pair, gate, dout)
    for b in range(B):
        for first in (0, N - 3):
            part = [t[b:b + 1, first:first + 3].contiguous() for t in (q, k, v, gate, dout)]
            small = _gradients(part[0], part[1], part[2], pair[b:b + 1], part[3], part[4])
            for name, x, y in zip(("out", "dq", "dk", "dv", "dgate"), large, small):
                assert torch.equal(x[b:b + 1, first:first + 3], y), (name, b, first)
    _check_pair_gradient(large[5], q, k, v, pair, (dout.double() * torch.sigmoid(gate.double())))


@pytest.mark.parametrize("N,S,H,D,row", [(161, 259, 8, 32, False), (97, 450, 8, 32, True), (101, 256, 7, 64, False)])
def test_layouts_of_calls_that_touch_rows_ahead(N, S, H, D, row):
    """Operands and an output gradient that are parts of wider tensors, heads first, or the same for every entry: what they are as copies."""
    g = torch.Generator(device=DEV).manual_seed(S)
    randn = lambda *shape: torch.randn(*shape, generator=g, device=DEV).bfloat16()  # noqa: E731
    pair = randn(1, H, S, S)
    biases = [(pair, N)] + ([(randn(N, 1, 1, S), 1)] if row else [])
    packed, wide = randn(N + 3, S, H, 3 * D), randn(N, H + 2, S, D)
    offset = [packed[2:N + 2, :, :, i * D:(i + 1) * D].transpose(1, 2) for i in range(3)]      # of one projection, the first entries left out
    cases = [(*offset, randn(N, S, H, D).transpose(1, 2)),
             (wide[:, 1:H + 1], randn(N, H, S + 5, D)[:, :, 5:], randn(N, H, S, 2 * D)[..., D:], wide.flip(0)[:, 2:]),
             (randn(1, H, S, D).expand(N, H, S, D), randn(N, 1, S, D).expand(N, H, S, D), offset[0], randn(1, H, S, D).expand(N, H, S, D)),
             (offset[1], offset[2], randn(1, 1, S, D).expand(N, H, S, D), randn(N, H, 1, D).expand(N, H, S, D))]
    for q, k, v, dout in cases:
        results = []
        for made in (lambda t: t.detach(), lambda t: t.detach().contiguous()):
            leaves = [made(t).requires_grad_(True) for t in (q, k, v, pair)]
            out = ops.dispatch(*leaves[:3], biases=[(leaves[3], N)] + biases[1:])
            results.append([out.detach(), *torch.autograd.grad(out, leaves, made(dout))])
        for name, a, b in zip(("out", "dq", "dk", "dv", "dbias"), *results):
            assert torch.equal(a, b), name
