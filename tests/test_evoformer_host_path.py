"""The Evoformer front end's native path (csrc/host.cpp `evoformer`) against the front end's own views and ops.dispatch."""
import pytest
import torch

from flashlight_amd import _ffi
from flashlight_amd.attention_variants import attention_reference
from tests.test_host_path import _same

DEV = "cuda"


class _Views:
    """The native module without the Evoformer entry: the front end makes the 4-D views, ops.dispatch goes on natively."""

    def __init__(self, host):
        self.forward, self.key_chunks = host.forward, host.key_chunks

    def evoformer(self, *args):
        return None


def _both(monkeypatch, run):
    native = run()
    with monkeypatch.context() as m:
        m.setattr(_ffi, "_host", _Views(_ffi._host))
        return native, run()


def _counting(monkeypatch, taken):
    host = _ffi._host

    class Counting(_Views):
        def evoformer(self, *args):
            out = host.evoformer(*args)
            taken.append(out is not None)
            return out
    monkeypatch.setattr(_ffi, "_host", Counting(host))


def _layouts(lead, S, H, D, dtype):
    g = torch.Generator().manual_seed(S)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)  # noqa: E731
    yield "contiguous", [r(*lead, S, H, D) for _ in range(4)], True
    yield "projection", list(r(*lead, S, 4, H, D).unbind(-3)), True
    yield "heads first", [r(*lead, H, S, D).transpose(-2, -3) for _ in range(4)], True
    yield "one row for all", [r(*lead, S, H, D)] + [r(S, H, D).expand(*lead, S, H, D) for _ in range(3)], True
    yield "off by one element", [r(*lead, S, H, D + 8)[..., 1:D + 1] for _ in range(4)], False
    if len(lead) > 1:  # (leading axes that do not merge into one, unless one of them is 1)
        yield "swapped leading axes", [r(lead[1], lead[0], *lead[2:], S, H, D).transpose(0, 1) for _ in range(4)], 1 in lead


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lead,S,H,D", [((6,), 64, 2, 32), ((2, 3), 70, 2, 32), ((1, 5), 33, 1, 64), ((2, 1, 4), 40, 4, 64)])
def test_layouts_and_biases(lead, S, H, D, dtype, monkeypatch):
    _ffi.load_library()
    g = torch.Generator().manual_seed(len(lead))
    r = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)  # noqa: E731
    one = (1,) * (len(lead) - 1)
    pairs = [r(lead[0], *one, H, S, S), r(*(1,) * len(lead), H, S, S), r(H, S, S), torch.randn(H, S, S, generator=g).to(DEV),
             r(H, S, S + 8)[..., :S]]
    mask = torch.where(torch.rand(*lead, 1, 1, S, generator=g) < 0.2, -6e4, 0.0).to(dtype).to(DEV)
    taken = []
    _counting(monkeypatch, taken)
    for name, (q, k, v, gate), native in _layouts(lead, S, H, D, dtype):
        for i, pair in enumerate(pairs):
            for kw in ({}, {"gate": gate}):
                biases = [[pair], [mask, pair], [pair, mask]][i % 3]
                del taken[:]
                run = lambda: [attention_reference(q, k, v, biases, **kw)]  # noqa: E731
                _same(*_both(monkeypatch, run))
                assert taken == [native], name
                leaves = [t.detach().requires_grad_(True) for t in (q, k, v, pair, *kw.values())]
                p = leaves[3]
                biases = [[p], [mask, p], [p, mask]][i % 3]
                kw = {"gate": leaves[4]} if kw else {}
                out = attention_reference(*leaves[:3], biases, **kw)
                assert out.shape == q.shape
                flat = r(*lead, S, H, D)
                for dout in (flat, flat.transpose(-2, -3).contiguous().transpose(-2, -3), flat[..., :1].expand_as(flat),
                             r(*lead, S, H, D + 3)[..., 1:D + 1]):
                    def grads():
                        out = attention_reference(*leaves[:3], biases, **kw)
                        return [out.detach(), *torch.autograd.grad(out, leaves, dout)]
                    if pair.dtype == dtype or lead != (1, 5):  # (one bias per batch entry of one: not shared, summed another way)
                        _same(*_both(monkeypatch, grads))


@pytest.mark.gpu
def test_what_it_leaves_to_the_front_end(monkeypatch):
    """Calls that are refused, converted or composed there: the same results and errors as ever."""
    _ffi.load_library()
    taken = []
    _counting(monkeypatch, taken)
    g = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)  # noqa: E731
    q, k, v, pair, row = r(2, 3, 20, 2, 32), r(2, 3, 20, 2, 32), r(2, 3, 20, 2, 32), r(2, 1, 2, 20, 20), r(2, 3, 1, 1, 20)
    calls = [(q, k, v, [pair, row, row]), (q, k, v, [r(3, 2, 20, 20)]), (q, k, v, [r(2, 1, 2, 20, 1)]),
             (q[..., :24], k[..., :24], v[..., :24], [pair]), (q, k[:, :, :10], v[:, :, :10], []), (q[:0], k[:0], v[:0], [])]
    for args in calls:
        _same(*_both(monkeypatch, lambda: [attention_reference(*args)]))
    assert not any(taken)
    for args, error in (((q, k[:, :, :10], v[:, :, :10], [pair]), ValueError), ((q, k, v, [r(2, 1, 3, 20, 20)]), ValueError),
                        ((q, k, v, [r(1, 2, 1, 2, 20, 20)]), ValueError), ((q[0, 0], k[0, 0], v[0, 0], []), ValueError)):
        with pytest.raises(error):
            attention_reference(*args)


@pytest.mark.gpu
def test_autograd_around_the_node(monkeypatch):
    """Hooks on saved tensors, in-place changes of operands and result, partial gradients, a second derivative."""
    _ffi.load_library()
    g = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)  # noqa: E731
    leaves = [r(1, 4, 70, 2, 32).requires_grad_(True) for _ in range(3)] + [r(1, 1, 2, 70, 70).requires_grad_(True)]
    gate, dout = r(1, 4, 70, 2, 32).requires_grad_(True), r(1, 4, 70, 2, 32)
    for kw in ({}, {"gate": gate}):
        run = lambda q, k, v, p: attention_reference(q, k, v, [p], **kw)  # noqa: E731
        want = torch.autograd.grad(run(*leaves), leaves, dout)
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.to(DEV)):
            out = run(*leaves)
        _same(torch.autograd.grad(out, leaves, dout), want)
        assert len(packed) >= 6
        _same(torch.autograd.grad(run(*leaves[:3], leaves[3].detach()), leaves[:3], dout), want[:3])
        _same(torch.autograd.grad(run(*(t.detach() for t in leaves[:3]), leaves[3]), leaves[3:], dout), want[3:])
        for change in (0, 3):
            x = [t * 1.0 for t in leaves]
            out = run(*x)
            with torch.no_grad():
                x[change].add_(1.0)
            with pytest.raises(RuntimeError, match="modified by an inplace operation"):
                torch.autograd.grad(out, leaves, dout)
        if not kw:  # (under a gate the gradients do not need the gated result)
            out = run(*leaves)
            with torch.no_grad():
                out.add_(1.0)
            with pytest.raises(RuntimeError, match="modified by an inplace operation"):
                torch.autograd.grad(out, leaves, dout)
        dq, = torch.autograd.grad(run(*leaves).float().sum(), leaves[:1], create_graph=True)
        with pytest.raises(RuntimeError, match="not differentiable a second time"):
            dq.float().sum().backward()
