"""Document-mask forwards whose workgroups list their key tiles themselves (doc_own in csrc/fwd_kernel.h): the lists of the launch they
stand in for, at the edges of 64 tiles, for ids of any order and size; workspaces they prepared, read by calls of any size."""
import pytest
import torch

from flashlight_amd import _ffi
from tests.test_abi import good_params

DEV = "cuda"
KINDS = ("sorted", "unsorted", "huge", "one", "pairs")


def _ids(kind, B, S, g):
    if kind == "one":
        return torch.full((B, S), -7, dtype=torch.int64)
    if kind == "pairs":
        return torch.arange(S).repeat(B, 1) // 2
    ids = torch.randint(-3, 4, (B, S), generator=g)
    return ids.sort(dim=1).values if kind == "sorted" else ids * 2 ** 40 + (1 << 33) if kind == "huge" else ids


@pytest.mark.gpu
@pytest.mark.parametrize("mask", [_ffi.MASK_DOCUMENT, _ffi.MASK_DOCUMENT_CAUSAL])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("S", [1, 31, 33, 64, 129, 700, 4096, 4097])
def test_own_lists_are_those_of_the_launch(S, kind, mask):
    """Head dim 32 has one form of the kernel: a call of many workgroups, whose lists are made by a launch, gives the same bits."""
    g = torch.Generator().manual_seed(S)
    ids = _ids(kind, 2, S, g).to(DEV)
    q, k, v = (torch.randn(2, 2, S, 32, generator=g).to(torch.bfloat16).to(DEV) for _ in range(3))
    out = _ffi.attn_fwd(q, k, v, mask_kind=mask, doc_ids=ids)
    times = 1024 // (2 * -(-S // 128)) + 1
    many = _ffi.attn_fwd(*(t.repeat(1, times, 1, 1) for t in (q, k, v)), mask_kind=mask, doc_ids=ids)
    assert torch.equal(out, many[:, :2]) and torch.equal(out, many[:, -2:])


@pytest.mark.gpu
@pytest.mark.parametrize("D,S", [(64, 600), (128, 2048), (128, 2049), (64, 1)])
def test_prepared_workspaces_serve_calls_of_other_heads(D, S):
    """What a call of few workgroups leaves in the workspace has lists but no order of the query tiles; calls of many workgroups read
    it all the same, and the other way round."""
    g = torch.Generator().manual_seed(D + S)
    ids = torch.randint(0, 5, (2, S), generator=g).sort(dim=1).values.to(DEV)
    few, many = 2, 600 // -(-S // 128) + 1
    operands = {H: tuple(torch.randn(2, H, S, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(3)) for H in (few, many)}
    plain = {H: _ffi.attn_fwd(*x, mask_kind=_ffi.MASK_DOCUMENT_CAUSAL, doc_ids=ids) for H, x in operands.items()}
    for first, then in ((few, many), (many, few), (few, few)):
        ws = _ffi.DocWorkspace()
        for H in (first, then):
            if ws.key is not None:  # the C interface does not ask for the same heads; the Python handle does
                ws.key = ws.key[:5] + (H, H) + ws.key[7:]
            q, k, v = operands[H]
            ready = ws.buffer
            out = _ffi.attn_fwd(q, k, v, mask_kind=_ffi.MASK_DOCUMENT_CAUSAL, doc_ids=ids, doc_workspace=ws)
            assert ready is None or ws.buffer is ready  # (not prepared anew)
            assert torch.equal(out, plain[H]), (first, then, H)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["sorted", "falling", "scattered"])
@pytest.mark.parametrize("S", [8193, 20000, 32768, 32769, 66001])  # the order in the lists' launch up to 256 query tiles, then in one of its own
def test_every_query_tile_has_a_place_in_the_order(S, kind):
    """Documents of two positions: a row's result is its value, or the softmax of two logits over two values."""
    H, D, pairs = 4, 64, (S + 1) // 2
    g = torch.Generator().manual_seed(S)
    q, k, v = (torch.randn(1, H, S, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(3))
    number = torch.arange(S) // 2
    ids = {"sorted": number, "falling": -number, "scattered": number * 7919 % pairs}[kind]
    out = _ffi.attn_fwd(q, k, v, mask_kind=_ffi.MASK_DOCUMENT_CAUSAL, doc_ids=ids[None].to(DEV)).double()
    qd, kd, vd = q.double(), k.double(), v.double()
    even, odd = slice(0, None, 2), slice(1, None, 2)
    assert torch.equal(out[:, :, even], vd[:, :, even])
    n = S // 2
    logits = torch.stack([(qd[:, :, odd] * kd[:, :, even][:, :, :n]).sum(-1), (qd[:, :, odd] * kd[:, :, odd]).sum(-1)], -1) * D ** -0.5
    w = logits.softmax(-1)
    want = w[..., :1] * vd[:, :, even][:, :, :n] + w[..., 1:] * vd[:, :, odd]
    # weights rounded to 16 bits, numerator and row sum alike, and one rounding of the result
    bound = 2.0 ** -8 * (w[..., :1] * vd[:, :, even][:, :, :n].abs() + w[..., 1:] * vd[:, :, odd].abs() + 2 * want.abs())
    assert ((out[:, :, odd] - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("mask", [_ffi.MASK_DOCUMENT, _ffi.MASK_DOCUMENT_CAUSAL])
@pytest.mark.parametrize("kind", ["sorted", "shuffled", "scattered"])
@pytest.mark.parametrize("B,S,D", [(1, 8193, 64), (3, 8100, 64), (2, 8193, 32), (4, 8193, 64), (1, 32768, 128), (1, 32769, 128), (1, 66001, 64), (2, 70000, 32)])
def test_query_tiles_are_dealt_by_falling_length(B, S, D, kind, mask):
    """The order that the pre-pass leaves behind the lists: every query tile once, by falling number of key tiles, whatever the ids.  The launch
    that finds it beside the lists counts tiles against the ids of the whole query tile: its lengths may be longer than the lists."""
    g = torch.Generator().manual_seed(S)
    lengths = torch.randint(20, 900, (S // 20,), generator=g)
    number = torch.arange(len(lengths)) if kind == "sorted" else torch.randperm(len(lengths), generator=g)
    ids = torch.repeat_interleave(number, lengths)[:S]
    if kind == "scattered":
        ids = (ids * 7919 + torch.arange(S) // 3000 % 2 * torch.randint(0, 9, (S,), generator=g)) % len(lengths)
    ids = torch.stack([ids.roll(b * 700) if kind != "sorted" else ids + (ids > 5 * b).long() for b in range(B)]).to(DEV)
    q = torch.zeros(B, 1 if D == 128 else 2 if B * S > 60000 else 8, S, D, dtype=torch.bfloat16, device=DEV)
    ws = _ffi.DocWorkspace()
    _ffi.attn_fwd(q, q, q, mask_kind=mask, doc_ids=ids, doc_workspace=ws)
    words = ws.buffer.view(torch.int32).cpu()
    p = good_params(B=B, Hq=q.shape[1], Hkv=q.shape[1], L=S, D=D)
    p.mask_kind, p.doc_ids, p.doc_stride, p.workspace, p.workspace_bytes = mask, 0x50000, S, 0x60000, ws.buffer.numel()
    plan = _ffi.plan(p)
    bm, bn = plan["rows_per_workgroup"], plan["keys_per_tile"]
    tiles, nk = -(-S // bm), -(-S // bn)
    stride, table = -(-(nk + 1) // 4) * 4, B * -(-S // 32) * 4
    listed = words[table:table + B * tiles * stride].view(B, tiles, stride)[:, :, 0].long()
    order = words[table + B * tiles * stride:][:B * tiles].view(B, tiles).long()
    assert torch.equal(order.sort(dim=1).values, torch.arange(tiles).expand(B, tiles))
    # key tiles whose ids meet those of the query tile's key tiles, up to the diagonal under the causal mask
    of_keys = torch.cat([ids.cpu(), ids.cpu()[:, -1:].expand(B, nk * bn - S)], 1).view(B, nk, bn)
    least, most = of_keys.min(-1).values, of_keys.max(-1).values
    per = bm // bn
    counted = torch.empty(B, tiles, dtype=torch.long)
    for t in range(tiles):
        first, last = t * per, min(t * per + per, nk) - 1
        lo, hi = least[:, first:last + 1].min(1, keepdim=True).values, most[:, first:last + 1].max(1, keepdim=True).values
        meets = (most >= lo) & (least <= hi)
        counted[:, t] = (meets[:, :last + 1] if mask == _ffi.MASK_DOCUMENT_CAUSAL else meets).sum(1)
    beside = tiles >= 64 and B * tiles <= 256  # (doc_orders in csrc/api.hip)
    dealt = (counted if beside else listed).gather(1, order)
    assert (dealt[:, 1:] <= dealt[:, :-1]).all()
    assert (listed <= counted).all()
