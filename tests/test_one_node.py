"""The native layer calls under callers that record what Python runs (quartet_amd/one_node.py), without a GPU: a stand-in for
the native extension whose results PyTorch's operators did not compute, as a kernel's are not."""
import warnings

import pytest
import torch
from torch.autograd import forward_ad

import quartet_amd as q
from quartet_amd import _lib
from quartet_amd.one_node import as_one_node


class _Host:
    """Results written behind the back of PyTorch's operators into memory they allocated."""

    @staticmethod
    def _opaque(x, w):
        y = torch.empty(x.shape[0], w.shape[0])
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")
            y.detach().numpy()[:] = x.detach().numpy() @ w.detach().numpy().T
        return y

    def linear(self, x, weight, *rest):
        return self._opaque(x, weight), None

    def quantizer(self, x, hd, signs, mode, seed, post):
        return self._opaque(x, torch.eye(x.shape[1]) * (3.0 + seed % 2))


@pytest.fixture
def host(monkeypatch):
    monkeypatch.setattr(_lib, "host", _Host)


def _layer():
    torch.manual_seed(0)
    return q.QuantizedLinear(64, 32, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(), activation_quantizer=q.QuestMXFP4Quantizer(),
                             gradient_quantizer=q.AlbertTsengQuantizer(), backward_scheme=q.BACKWARD_SCHEMES["Q(E)Q(Wt)t_Q(Et)Q(Xt)t"]())


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("make", [_layer, q.QuestMXFP4Quantizer, lambda: q.AlbertTsengQuantizer(stochastic=False)])
def test_a_trace_runs_the_call_again(host, make):
    module = make()
    with torch.no_grad():
        traced = torch.jit.trace(module, (torch.randn(8, 64),), check_trace=False)
        for seed in range(3):
            x = torch.randn(8, 64, generator=torch.Generator().manual_seed(seed))
            assert torch.equal(traced(x), module(x))


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("filled", [False, True])
def test_a_trace_follows_the_weight(host, filled):
    """A replay looks the packed weight up again: nothing of the traced call's weight is kept."""
    layer = _layer()
    q.enable_packed_weight_cache(layer)
    x = torch.randn(8, 64)
    with torch.no_grad():
        if filled:
            layer(x)
        traced = torch.jit.trace(layer, (x,), check_trace=False)
        layer.weight.mul_(-2.0)
        assert torch.equal(traced(x), layer(x))


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("make", [_layer, q.QuestMXFP4Quantizer, lambda: q.AlbertTsengQuantizer(stochastic=False)])
def test_tangents_are_refused(host, make, grad):
    """No forward-mode derivative exists: a dual input or weight raises, also where nothing asks for a gradient; plain
    tensors go through at a dual level."""
    module = make()
    x = torch.randn(8, 64)
    with forward_ad.dual_level(), torch.set_grad_enabled(grad):
        with pytest.raises(NotImplementedError):
            module(forward_ad.make_dual(x, torch.ones_like(x)))
        if isinstance(module, q.QuantizedLinear):
            dual = forward_ad.make_dual(module.weight.detach(), torch.ones_like(module.weight))
            with pytest.raises(NotImplementedError):
                torch.func.functional_call(module, {"weight": dual}, (x,))
            module.requires_grad_(False)
        assert torch.equal(module(x), make()(x))


@pytest.mark.parametrize("make", [_layer, q.QuestMXFP4Quantizer])
def test_function_transforms_are_refused(host, make):
    module, x = make().requires_grad_(False), torch.randn(4, 8, 64)
    for transform in (lambda: torch.func.vmap(module)(x), lambda: torch.func.grad(lambda t: module(t).sum())(x[0]),
                      lambda: torch.func.jvp(module, (x[0],), (x[0],)), lambda: torch.func.vjp(module, x[0])):
        with pytest.raises(RuntimeError, match="functorch"):
            transform()


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
def test_a_trace_is_differentiable():
    """Two outputs, one of them left out of the loss, an argument that is no tensor, and one without a gradient."""
    @as_one_node
    def call(x, add, factor):
        y = x * x * factor + add
        return y, x * 5.0

    def net(x, add):
        return call(x, add, 3.0)
    x, add = torch.randn(4, 6).requires_grad_(True), torch.randn(4, 6)
    traced = torch.jit.trace(net, (x, add), check_trace=False)
    assert not any(node.kind() == "prim::Constant" and node.output().type().kind() == "TensorType" for node in traced.graph.nodes())
    for pick in (0, 1, None):
        a, b = (torch.randn(4, 6, generator=torch.Generator().manual_seed(5)).requires_grad_(True) for _ in range(2))
        for t, f in ((a, traced), (b, net)):
            out = f(t, add)
            ((out[0] + out[1]) if pick is None else out[pick]).sum().backward()
        assert torch.equal(a.grad, b.grad)
    y, _ = traced(a, add)
    y.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        y.sum().backward()
