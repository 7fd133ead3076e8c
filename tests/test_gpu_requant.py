"""The backward pass's re-quantizer (rotation on the matrix pipe) against the stand-alone operators: a layer's gradients, bit for
bit, equal what quantizers, re-quantizers, products and inverse rotations give when they are called one by one on row-major
operands.  Rows of x and W whose scales spread over more octaves than the matrix instruction adds exactly take another route."""
import random

import pytest
import torch

from quartet_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("shape", [(128, 128, 128), (640, 256, 384), (1152, 192, 320), (160, 96, 224)])
@pytest.mark.parametrize("spread", [0, 9, 12, 40])
@pytest.mark.parametrize("stochastic", [True, False])
def test_gradients_equal_the_operators_one_by_one(hd, shape, spread, stochastic):
    import quartet_amd as q
    T, I, O = (max(hd, n // hd * hd) for n in shape)
    print(f"case requant hd={hd} shape={(T, I, O)} spread={spread} stochastic={stochastic}", flush=True)
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(spread + hd)
    exponents = lambda n: (torch.rand(n, 1, generator=g) * (spread + 1)).floor() - spread // 2
    x = torch.randn(T, I, generator=g) * torch.exp2(exponents(T))
    w = 0.02 * torch.randn(O, I, generator=g) * torch.exp2(exponents(O).clamp(-4, 4))
    if spread:
        x[5::37] = 0   # zero rows: the smallest scale a quest quantizer writes
    x, w, e = x.to(dev, torch.bfloat16), w.to(dev, torch.bfloat16), (1e-3 * torch.randn(T, O, generator=g)).to(dev, torch.bfloat16)
    layer = q.QuantizedLinear(I, O, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(hadamard_dim=hd),
                              activation_quantizer=q.QuestMXFP4Quantizer(hadamard_dim=hd),
                              gradient_quantizer=q.AlbertTsengQuantizer(hadamard_dim=hd, stochastic=stochastic, rerotate="signs"),
                              backward_scheme=q.BACKWARD_SCHEMES["Q(E)Q(Wt)t_Q(Et)Q(Xt)t"]()).to(dev, torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(w)
    xd = x.clone().requires_grad_(True)
    torch.manual_seed(3)
    random.seed(17)
    layer(xd).backward(e)
    random.seed(17)
    seeds = [random.getrandbits(63) for _ in range(4)] if stochastic else [0] * 4
    signs = layer.backward_scheme.g_quantizer.sign_bits
    mode = K.QM_ABSMAX_SR if stochastic else K.QM_ABSMAX_RTN
    alpha = float(torch.tensor(K.FOUR_THIRDS, dtype=torch.float32) * torch.tensor(K.FOUR_THIRDS, dtype=torch.float32))
    xc, xs, xm, _ = K.quantize_mxfp4(x, hd, None, K.QM_QUEST_RTN, want_mask=True)
    wc, ws, wm, _ = K.quantize_mxfp4(w, hd, None, K.QM_QUEST_RTN, want_mask=True)
    ec, es, _, _ = K.quantize_mxfp4(e, hd, signs, mode, seed=seeds[0])
    wtc, wts, _ = K.requantize_transposed_mxfp4(wc, ws, 1.0, torch.bfloat16, hd, signs, mode, seed=seeds[1])
    etc, ets, _, _ = K.quantize_mxfp4(e, hd, signs, mode, transposed_in=True, seed=seeds[2])
    xtc, xts, _ = K.requantize_transposed_mxfp4(xc, xs, 1.0, torch.bfloat16, hd, signs, mode, seed=seeds[3])
    gx = K.masked_hadamard_bwd(K.gemm_mxfp4_tn(ec, es, wtc, wts, alpha, torch.bfloat16), hd, torch.bfloat16, None, xm)
    gw = K.masked_hadamard_bwd(K.gemm_mxfp4_tn(etc, ets, xtc, xts, alpha, torch.bfloat16), hd, torch.bfloat16, None, wm)
    assert torch.equal(xd.grad, gx)
    assert torch.equal(layer.weight.grad, gw)
