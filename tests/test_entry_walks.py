"""The shared-bias kernels' walks over batch entries: the order of workgroups with the heads of a chunk on one XCD, and rows touched ahead of
their transfers in the gradients of calls whose operands are larger than the caches (csrc/tile_operands.h, pairbias_bwd_kernel.h).  Neither
changes a sum, so a part of the entries alone, which takes neither, has the same bits."""
import pytest
import torch

from flashlight_amd import attention_variants as A

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gradients(q, k, v, pair, gate, dout):
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v, gate, pair)]
    out = A.attention_reference(*leaves[:3], [leaves[4]], gate=leaves[3])
    return [out.detach(), *torch.autograd.grad(out, leaves, dout)]


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
    assert torch.isfinite(large[5]).all()
