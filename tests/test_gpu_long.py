"""Layers over more tokens than the tile kernels contract (2^23): the gradient of W sums over all of them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", ["Q(E)Q(Wt)t_Q(Et)Q(Xt)t", "Q(E)W_Q(Et)X"])
def test_layer_over_eight_million_tokens(scheme):
    import quartet_amd as q
    dev, T, I, O = torch.device("cuda:0"), 1 << 23, 64, 64
    print(f"case layer {T}x{I}x{O} {scheme}", flush=True)
    torch.manual_seed(0)
    layer = q.QuantizedLinear(I, O, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(), activation_quantizer=q.QuestMXFP4Quantizer(),
                              gradient_quantizer=q.AlbertTsengQuantizer(stochastic=False, rerotate="signs"),
                              backward_scheme=q.BACKWARD_SCHEMES[scheme](), device=dev, dtype=torch.bfloat16)
    q.enable_packed_weight_cache(layer)
    g = torch.Generator(device=dev).manual_seed(1)
    x = torch.randn(T, I, generator=g, device=dev, dtype=torch.bfloat16).requires_grad_(True)
    e = torch.randn(T, O, generator=g, device=dev, dtype=torch.bfloat16)
    y = layer(x)
    y.backward(e)
    gw, layer.weight.grad = layer.weight.grad, None
    # the same tokens in 32 calls: rows of y and of x's gradient are independent, W's gradient is the calls' sum up to one
    # bf16 rounding each (2^-9 relative)
    total = torch.zeros(O, I, device=dev)
    for rows in torch.arange(T, device=dev).view(32, -1)[:, [0, -1]].tolist():
        part = x.detach()[rows[0]:rows[1] + 1].requires_grad_(True)
        z = layer(part)
        z.backward(e[rows[0]:rows[1] + 1])
        for short, long in ((z.detach(), y.detach()), (part.grad, x.grad)):
            long = long[rows[0]:rows[1] + 1]
            if scheme == "Q(E)W_Q(Et)X":   # the long call runs on the module path: its operands and gradients are rounded to bf16 on the way
                assert float((short.float() - long.float()).norm() / short.float().norm()) < 1e-2
            else:
                assert torch.equal(short, long)
        total += layer.weight.grad.float()
        layer.weight.grad = None
    rel = float((gw.float() - total).norm() / total.norm())
    assert rel < 2.0 ** -7, rel
