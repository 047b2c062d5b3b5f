"""Which calls of a dense projection may go past the library's product."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD

from lfmq.models.linear import Linear
from lfmq.ops import functional as F


def test_values_only():
    """The kernels' binding knows tensors and threads that stand for more
    than values, by the ways that torch has for that."""
    plain = pytest.importorskip("lfmq_seq").values_only
    x = torch.randn(3, 4)
    seen = []

    def note(t):
        seen.append(plain(t))
        return t + 1

    assert plain(x) and plain(torch.nn.Parameter(x))
    with torch.inference_mode():
        assert plain(x) and plain(torch.randn(2))
    with torch.no_grad(), torch.device("cpu"), torch.autocast("cpu"):
        assert plain(x)
    with fwAD.dual_level():
        assert not plain(fwAD.make_dual(x, x))
    torch.func.vmap(note)(x)
    torch.func.jvp(note, (x,), (x,))
    torch.func.grad(lambda t: note(t).sum())(x)
    torch.jit.trace(note, (x,), check_trace=False)
    from torch.utils.flop_counter import FlopCounterMode
    with FlopCounterMode(display=False):
        note(x)
    from torch._subclasses import FakeTensorMode
    with FakeTensorMode():
        note(torch.randn(2))
    assert seen == [False] * 6
    assert not plain(torch._neg_view(x)) and not plain(x.to_sparse())
    assert plain(x)


def test_plain_tensors():
    class Sub(torch.Tensor):
        pass

    x, w = torch.randn(3, 4), torch.nn.Parameter(torch.randn(5, 4))
    with torch.no_grad():
        assert F._plain(x, w) and F._plain(x, w.detach())
        assert not F._plain(x, torch.nn.Parameter(w.detach().as_subclass(Sub)))
        assert not F._plain(x.as_subclass(Sub), w)
        with torch.device("cpu"):
            assert F._plain(x, w)

        class Mode(torch.overrides.TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                return func(*args, **(kwargs or {}))

        with Mode():
            assert not F._plain(x, w)
    assert not F._plain(x, w)


def test_projection_is_traced_as_the_library_s_product():
    m = Linear(4, 5, torch.float32)
    x = torch.randn(3, 4)
    g = torch.fx.symbolic_trace(m)
    assert any(n.target is torch.nn.functional.linear for n in g.graph.nodes)
    assert torch.equal(g(x), m(x))
    with torch.no_grad():
        c = torch.compile(m, backend="eager", fullgraph=True)
        assert torch.equal(c(x), m(x))
    assert torch.equal(torch.func.vmap(m)(x), torch.func.vmap(
        lambda v: torch.nn.functional.linear(v, m.weight))(x))
