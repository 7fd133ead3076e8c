"""The two gradient products of a layer in one launch, against the same products launched one by one."""
import re

import pytest
import torch

from tests.test_kernel_resources import kernels  # noqa: F401  (a fixture)
from tests.util import make_input

pytestmark = pytest.mark.gpu

QM_LAYOUT_PADDED = 2
ALPHA = float(torch.tensor(4.0 / 3.0, dtype=torch.float32) ** 2)


# K steps in whole blocks of four and not (muted ones), either product the long one, as many K steps; tiles over the edges of M and N by
# multiples of 64 and 32 rows; numbers of tiles that the XCDs and their workgroups share evenly and not, fewer long tiles than workgroups
@pytest.mark.parametrize("T,I,O", [(4096, 2048, 4096), (5888, 4800, 1536), (3168, 1984, 4800), (2944, 5440, 2080), (2016, 5312, 4096), (6144, 3072, 3072)])
@pytest.mark.parametrize("gx_rotated,gw_dtype", [(False, torch.bfloat16), (False, torch.float32), (True, torch.bfloat16), (True, torch.float32)])
def test_gradients_in_one_launch(monkeypatch, T, I, O, gx_rotated, gw_dtype):
    check_gradients(monkeypatch, T, I, O, 32, gx_rotated, gw_dtype, 1, 0x5A5A5A5A, 0x0F0F1234)


# blocks of 64 and 128 in the epilogue of one launch and (14464 x 576 x 1024) of two, with column signs that repeat every 32 and with others, which that epilogue does not take
@pytest.mark.parametrize("T,I,O,hd,path", [(2560, 2560, 5248, 128, 1), (2560, 3584, 5728, 128, 1), (1216, 4608, 4352, 64, 1), (3168, 1984, 4800, 64, 1), (14464, 576, 1024, 64, 0)])
@pytest.mark.parametrize("gw_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("repeat", [True, False])
def test_wider_blocks(monkeypatch, T, I, O, hd, path, gw_dtype, repeat):
    if not repeat and path == 1:   # the smaller tiles', or two launches
        path = None
    signs = [sum((s if repeat else s * 3 ** j & 0xFFFFFFFF) << 32 * j for j in range(hd // 32)) for s in (0x5A5A5A5A, 0x0F0F1234)]
    check_gradients(monkeypatch, T, I, O, hd, False, gw_dtype, path, *signs)


# the smaller tiles: either product the long one, four K steps and many, 128 x 128 and 64 x 64 of either product (paths as chosen now),
# ragged rows and columns, as many tiles as there are CUs and a handful; Hadamard blocks of every width
@pytest.mark.parametrize("T,I,O,hd", [(512, 640, 1920, 32), (1792, 1152, 2560, 32), (640, 4096, 8192, 32), (1888, 1664, 3584, 32), (4128, 1088, 4128, 32), (1024, 1056, 1536, 32),
                                      (8192, 512, 2048, 64), (2304, 1408, 2048, 64), (2304, 768, 3200, 128), (480, 2048, 8832, 32), (9216, 512, 9216, 32)])
@pytest.mark.parametrize("gw_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("gx_rotated", [False, True])
def test_gradients_in_one_launch_of_small_tiles(monkeypatch, T, I, O, hd, gx_rotated, gw_dtype):
    if gx_rotated and hd != 32:
        pytest.skip("rotated gradients are those of blocks of 32")
    signs = [sum((s * 3 ** j & 0xFFFFFFFF) << 32 * j for j in range(hd // 32)) for s in (0x5A5A5A5A, 0x0F0F1234)]
    check_gradients(monkeypatch, T, I, O, hd, gx_rotated, gw_dtype, 2, *signs)


def check_gradients(monkeypatch, T, I, O, hd, gx_rotated, gw_dtype, path, sx, sw):
    """Both kernels round the fp32 sums of the same K order to bf16, mask them and rotate them in fp32; the rotation's sums of 32 to 128
    values are in another order than the stand-alone kernel's (2^-24 of a group's norm apart), which turns a bf16 rounding now and
    then: at most one result in 10^4, by one step of 2^-8 of its value or, where a group cancels, 2^-20 of the group.  Without a
    rotation (gx_rotated) the bits are the same, and so are a wide gradient's and a bf16 one's; and all of them on the smaller tiles (path
    2), whose rotation is the stand-alone kernel's."""
    print(f"case pair {T}x{I}x{O} hd={hd} gx_rotated={gx_rotated} gw={gw_dtype}", flush=True)
    from quartet_amd import _lib, kernels as K
    if path is not None:
        assert _lib.lib().qm_linear_backward_in_one_launch(T, I, O, hd, hd, int(gw_dtype == torch.float32), int(gx_rotated)) == path
    monkeypatch.setattr(K, "_layout", lambda tiled: QM_LAYOUT_PADDED if tiled == "padded" else K.QM_LAYOUT_TILED if tiled else K.QM_LAYOUT_ROWMAJOR)
    dev, bf16 = "cuda:0", torch.bfloat16
    x = make_input(T, I, bf16, seed=21).to(dev)
    w = make_input(O, I, bf16, seed=22, scale=0.02).to(dev)
    e = make_input(T, O, bf16, seed=23, scale=1e-2, outlier_frac=0).to(dev)
    sg, seeds = 0x13572468, [11, 12, 13, 14]
    _, px, pw = K.linear_forward(x, w, hd, sx, hd, sw, bf16, "padded")
    call = lambda dtype: K.linear_backward(e, px, pw, T, I, O, hd, sx, hd, sw, 32, sg, K.QM_ABSMAX_SR, seeds, bf16, bf16, bf16, bf16, bf16,
                                           "padded", gx_rotated=gx_rotated, gw_dtype=dtype)
    gx, gw = call(gw_dtype)
    assert gx.dtype == bf16 and gw.dtype == gw_dtype
    again = call(gw_dtype)
    assert torch.equal(gx, again[0]) and torch.equal(gw, again[1])
    assert torch.equal(gw.float(), call(bf16)[1].float())
    xc, xs, xm, _ = K.quantize_mxfp4(x, hd, sx, K.QM_QUEST_RTN, want_mask=True)
    wc, ws, wm, _ = K.quantize_mxfp4(w, hd, sw, K.QM_QUEST_RTN, want_mask=True)
    ec, es, _, _ = K.quantize_mxfp4(e, 32, sg, K.QM_ABSMAX_SR, seed=seeds[0])
    wtc, wts, _ = K.requantize_transposed_mxfp4(wc, ws, 1.0, bf16, 32, sg, K.QM_ABSMAX_SR, seed=seeds[1])
    etc, ets, _, _ = K.quantize_mxfp4(e, 32, sg, K.QM_ABSMAX_SR, transposed_in=True, seed=seeds[2])
    xtc, xts, _ = K.requantize_transposed_mxfp4(xc, xs, 1.0, bf16, 32, sg, K.QM_ABSMAX_SR, seed=seeds[3])
    gxq = K.gemm_mxfp4_tn(ec, es, wtc, wts, ALPHA, bf16, split_k=False)
    gwq = K.gemm_mxfp4_tn(etc, ets, xtc, xts, ALPHA, bf16, split_k=False)
    if gx_rotated:
        assert torch.equal(gx, gxq)
    for got, product, signs, mask in [(gw, gwq, sw, wm)] + ([] if gx_rotated else [(gx, gxq, sx, xm)]):
        want = K.masked_hadamard_bwd(product, hd, bf16, signs, mask)
        if path == 2:
            assert torch.equal(got.float(), want.float())
        far = (got.float() - want.float()).abs()
        group = product.float().view(-1, hd).norm(dim=1).repeat_interleave(hd).view(want.shape)
        assert int((far > 0).sum()) <= want.numel() * 1e-4
        assert bool((far <= 2.0 ** -7 * want.float().abs() + 2.0 ** -20 * group).all())


# a weight gradient that launched by itself is cut into K ranges (whether it is, and by which kernel, is near the line of the choice),
# one that is not, one that two launches serve
@pytest.mark.parametrize("T,I,O", [(32768, 640, 3456), (16480, 1728, 640), (4096, 2048, 4608), (16384, 5504, 512)])
def test_a_fused_layer_has_the_unfused_ones_weight_gradient(monkeypatch, T, I, O):
    """Bit for bit, whether the input gradient is rotated back by its product or left rotated for the kernel behind it."""
    print(f"case weight gradient of fused and unfused {T}x{I}x{O}", flush=True)
    from quartet_amd import kernels as K
    monkeypatch.setattr(K, "_layout", lambda tiled: QM_LAYOUT_PADDED)
    dev, bf16 = "cuda:0", torch.bfloat16
    x = make_input(T, I, bf16, seed=21).to(dev)
    w = make_input(O, I, bf16, seed=22, scale=0.02).to(dev)
    e = make_input(T, O, bf16, seed=23, scale=1e-2, outlier_frac=0).to(dev)
    _, px, pw = K.linear_forward(x, w, 32, 0x5A5A5A5A, 32, 0x0F0F1234, bf16, True)
    grads = {}
    for rotated in (False, True):
        for dtype in (bf16, torch.float32):
            grads[rotated, dtype] = K.linear_backward(e, px, pw, T, I, O, 32, 0x5A5A5A5A, 32, 0x0F0F1234, 32, 0x13572468, K.QM_ABSMAX_SR, [11, 12, 13, 14],
                                                      bf16, bf16, bf16, bf16, bf16, True, gx_rotated=rotated, gw_dtype=dtype)[1]
    for dtype in (bf16, torch.float32):
        assert torch.equal(grads[False, dtype], grads[True, dtype])


def test_which_gradients_share_a_launch():
    """Two launches (0), one of the 256 x 256 kernel (1), one of smaller tiles (2)."""
    from quartet_amd import _lib
    pairs = _lib.lib().qm_linear_backward_in_one_launch
    assert pairs(4096, 2048, 4096, 32, 32, _lib.QM_BF16, 0) == 1
    assert pairs(4096, 2080, 4096, 32, 32, _lib.QM_BF16, 0) == 2     # in_features not a multiple of 64
    assert pairs(1024, 1024, 256, 32, 32, _lib.QM_BF16, 0) == 0      # two K steps
    assert pairs(4096, 2048, 4096, 32, 32, _lib.QM_F32, 3) == 0      # no rotation at all
    assert pairs(0, 2048, 4096, 32, 32, _lib.QM_BF16, 0) == 0 and pairs(4096, 2048, 4100, 32, 32, _lib.QM_BF16, 0) == 0
    assert pairs(4096, 2048, 4096, 48, 32, _lib.QM_BF16, 0) == 0 and pairs(4096, 2048, 4096, 32, 32, 7, 0) == 0


def test_pairs_keep_nothing_in_memory(kernels):
    """No kernel with two products spills: a tile runs 4 to 30 K steps."""
    pairs = {n: v for n, v in kernels.items() if "pair_kernel<" in n or re.search(r"big4_kernel<.*, [1-9], (true|false)>\(", n)}
    assert len(pairs) >= 20
    assert {n: v for n, v in pairs.items() if v[1]} == {}


@pytest.mark.parametrize("T,I,O", [(4064, 4000, 3872), (3360, 3936, 3840)])
def test_error_only_gradients_in_one_launch(oracle, T, I, O):
    """Tiles over every edge, either product with more of them, both widths of the widened operands: against float64, as two launches are."""
    from quartet_amd import _lib
    from tests.test_gpu_tiles import test_error_only_layer_with_both_widths_in_one_product as against_float64
    assert _lib.lib().qm_linear_backward_error_in_one_launch(T, I, O, 32, _lib.QM_BF16) == 1
    against_float64(oracle, T, I, O)


# a weight gradient of fp32 weights (widened in the kernel) and of bf16 ones, as the first product of the grid (more tokens than out-features) and as
# the second, every Hadamard block; tiles over the edges
@pytest.mark.parametrize("T,I,O", [(4096, 3840, 3968), (3968, 3840, 4096)])
@pytest.mark.parametrize("hd,wide", [(32, True), (64, False), (64, True), (128, False), (128, True)])
def test_error_only_gradients_of_every_form_in_one_launch(oracle, T, I, O, hd, wide):
    """Against float64 on the oracle's tensors, every row: a rounding of the product to bf16 (2^-9), whose fp32 sum may lie on the other side of
    a tie, and one of the rotation."""
    import random

    import numpy as np

    import quartet_amd as q
    from quartet_amd import _lib
    from tests.test_gpu_tiles import error_only_layer
    from tests.util import to_oracle
    print(f"case error-only pair {T}x{I}x{O} hd={hd} wide={wide}", flush=True)
    assert _lib.lib().qm_linear_backward_error_in_one_launch(T, I, O, hd, _lib.QM_F32 if wide else _lib.QM_BF16) == 1
    x = make_input(T, I, torch.bfloat16, seed=1, outlier_frac=0.01)
    w = make_input(O, I, torch.bfloat16, seed=2, outlier_frac=0, scale=0.02)
    e = make_input(T, O, torch.bfloat16, seed=3, outlier_frac=0, scale=1e-3)
    layer = error_only_layer(q, I, O, hd, torch.float32 if wide else torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(w.to("cuda:0"))
    xd = x.to("cuda:0").requires_grad_(True)
    random.seed(5)
    with torch.autocast("cuda", torch.bfloat16, enabled=wide):
        layer(xd).backward(e.to("cuda:0"))
    assert xd.grad.dtype == torch.bfloat16 and layer.weight.grad.dtype == (torch.float32 if wide else torch.bfloat16)
    random.seed(5)
    o, d = oracle, float(oracle.FOUR_THIRDS)
    qx = o.quantize(to_oracle(x), hd, mode=o.QUEST_RTN, want_mask=True)
    qw = o.quantize(to_oracle(w.float() if wide else w), hd, mode=o.QUEST_RTN, want_mask=True)
    qe = o.quantize(to_oracle(e), hd, mode=o.ABSMAX_SR, seed=random.getrandbits(63))
    qet = o.quantize(to_oracle(e), hd, mode=o.ABSMAX_SR, transposed_in=True, seed=random.getrandbits(63))
    on_gpu = lambda t, scale: torch.from_numpy(o.dequantize(t["codes"], t["scales"], scale)).to("cuda:0").double()
    parity = torch.tensor([[bin(i & j).count("1") & 1 for j in range(hd)] for i in range(hd)], device="cuda:0")
    H = torch.where(parity == 1, -1.0, 1.0).double() * float(torch.tensor(hd ** -0.5).to(torch.bfloat16))

    def rotated(p, mask):
        keep = torch.from_numpy(np.unpackbits(np.asarray(mask).reshape(p.shape[0], -1), axis=1, bitorder="little")).to("cuda:0")
        return ((p.to(torch.bfloat16).double() * keep).view(-1, hd) @ H).view(p.shape)
    for got, want in [(xd.grad, rotated(on_gpu(qe, d) @ on_gpu(qw, 1.0), qx["mask"])), (layer.weight.grad, rotated(on_gpu(qet, d) @ on_gpu(qx, 1.0), qw["mask"]))]:
        err = (got.double() - want).norm(dim=1) / want.norm(dim=1)
        assert float(err.max()) < 4e-3, float(err.max())


# forward quantizers over different Hadamard blocks: the smaller tiles rotate either product by its own
@pytest.mark.parametrize("T,I,O", [(512, 640, 1920), (1888, 1664, 3584), (2048, 2048, 1536)])
@pytest.mark.parametrize("hd_x,hd_w,gx_rotated", [(32, 64, False), (32, 128, False), (64, 32, False), (128, 64, False), (32, 64, True)])
@pytest.mark.parametrize("gw_dtype", [torch.bfloat16, torch.float32])
def test_different_blocks_in_one_launch(monkeypatch, T, I, O, hd_x, hd_w, gx_rotated, gw_dtype):
    """Bit for bit the products and the stand-alone rotations."""
    print(f"case pair of blocks {T}x{I}x{O} hd={hd_x}, {hd_w} gx_rotated={gx_rotated} gw={gw_dtype}", flush=True)
    from quartet_amd import _lib, kernels as K
    assert _lib.lib().qm_linear_backward_in_one_launch(T, I, O, hd_x, hd_w, int(gw_dtype == torch.float32), int(gx_rotated)) == 2
    monkeypatch.setattr(K, "_layout", lambda tiled: QM_LAYOUT_PADDED if tiled == "padded" else K.QM_LAYOUT_TILED if tiled else K.QM_LAYOUT_ROWMAJOR)
    dev, bf16 = "cuda:0", torch.bfloat16
    x = make_input(T, I, bf16, seed=21).to(dev)
    w = make_input(O, I, bf16, seed=22, scale=0.02).to(dev)
    e = make_input(T, O, bf16, seed=23, scale=1e-2, outlier_frac=0).to(dev)
    sx, sw, sg, seeds = 0x5A5A5A5A, 0x0F0F1234, 0x13572468, [11, 12, 13, 14]
    _, px, pw = K.linear_forward(x, w, hd_x, sx, hd_w, sw, bf16, "padded")
    gx, gw = K.linear_backward(e, px, pw, T, I, O, hd_x, sx, hd_w, sw, 32, sg, K.QM_ABSMAX_SR, seeds, bf16, bf16, bf16, bf16, bf16,
                               "padded", gx_rotated=gx_rotated, gw_dtype=gw_dtype)
    xc, xs, xm, _ = K.quantize_mxfp4(x, hd_x, sx, K.QM_QUEST_RTN, want_mask=True)
    wc, ws, wm, _ = K.quantize_mxfp4(w, hd_w, sw, K.QM_QUEST_RTN, want_mask=True)
    ec, es, _, _ = K.quantize_mxfp4(e, 32, sg, K.QM_ABSMAX_SR, seed=seeds[0])
    wtc, wts, _ = K.requantize_transposed_mxfp4(wc, ws, 1.0, bf16, 32, sg, K.QM_ABSMAX_SR, seed=seeds[1])
    etc, ets, _, _ = K.quantize_mxfp4(e, 32, sg, K.QM_ABSMAX_SR, transposed_in=True, seed=seeds[2])
    xtc, xts, _ = K.requantize_transposed_mxfp4(xc, xs, 1.0, bf16, 32, sg, K.QM_ABSMAX_SR, seed=seeds[3])
    gxq = K.gemm_mxfp4_tn(ec, es, wtc, wts, ALPHA, bf16, split_k=False)
    gwq = K.gemm_mxfp4_tn(etc, ets, xtc, xts, ALPHA, bf16, split_k=False)
    assert torch.equal(gx, gxq if gx_rotated else K.masked_hadamard_bwd(gxq, hd_x, bf16, sx, xm))
    assert torch.equal(gw.float(), K.masked_hadamard_bwd(gwq, hd_w, bf16, sw, wm).float())
