"""The two gradient products of a layer in one launch, against the same products launched one by one."""
import pytest
import torch

from tests.util import make_input

pytestmark = pytest.mark.gpu

QM_LAYOUT_PADDED = 2
ALPHA = float(torch.tensor(4.0 / 3.0, dtype=torch.float32) ** 2)


# K steps in whole blocks of four and not (muted ones), either product the long one, as many K steps; tiles over the edges of M and N by
# multiples of 64 and 32 rows; numbers of tiles that the XCDs and their workgroups share evenly and not, fewer long tiles than workgroups
@pytest.mark.parametrize("T,I,O", [(4096, 2048, 4096), (5888, 4800, 1536), (4128, 4096, 4128), (1696, 2816, 7680), (6624, 4608, 1024), (3456, 3712, 1280),
                                   (2112, 3392, 4896)])
@pytest.mark.parametrize("gx_rotated,gw_dtype", [(False, torch.bfloat16), (False, torch.float32), (True, torch.bfloat16), (True, torch.float32)])
def test_gradients_in_one_launch(monkeypatch, T, I, O, gx_rotated, gw_dtype):
    check_gradients(monkeypatch, T, I, O, 32, gx_rotated, gw_dtype, True, 0x5A5A5A5A, 0x0F0F1234)


# blocks of 64 and 128 in the epilogue of one launch and of two (16384 x 2048 x 2048: the input gradient by itself, the weight gradient
# cut), with column signs that repeat every 32 and with others, which that epilogue does not take
@pytest.mark.parametrize("T,I,O,hd,paired", [(4096, 2048, 4096, 128, True), (4160, 2112, 4096, 64, True), (2048, 4096, 4224, 128, True), (16384, 2048, 2048, 64, False)])
@pytest.mark.parametrize("gw_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("repeat", [True, False])
def test_wider_blocks(monkeypatch, T, I, O, hd, paired, gw_dtype, repeat):
    signs = [sum((s if repeat else s * 3 ** j & 0xFFFFFFFF) << 32 * j for j in range(hd // 32)) for s in (0x5A5A5A5A, 0x0F0F1234)]
    check_gradients(monkeypatch, T, I, O, hd, False, gw_dtype, paired, *signs)


def check_gradients(monkeypatch, T, I, O, hd, gx_rotated, gw_dtype, paired, sx, sw):
    """Both kernels round the fp32 sums of the same K order to bf16, mask them and rotate them in fp32; the rotation's sums of 32 to 128
    values are in another order than the stand-alone kernel's (2^-24 of a group's norm apart), which turns a bf16 rounding now and
    then: at most one result in 10^4, by one step of 2^-8 of its value or, where a group cancels, 2^-20 of the group.  Without a
    rotation (gx_rotated) the bits are the same, and so are a wide gradient's and a bf16 one's."""
    print(f"case pair {T}x{I}x{O} hd={hd} gx_rotated={gx_rotated} gw={gw_dtype}", flush=True)
    from quartet_amd import _lib, kernels as K
    assert _lib.lib().qm_linear_backward_in_one_launch(T, I, O, hd, hd, int(gw_dtype == torch.float32), int(gx_rotated)) == paired
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
        far = (got.float() - want.float()).abs()
        group = product.float().view(-1, hd).norm(dim=1).repeat_interleave(hd).view(want.shape)
        assert int((far > 0).sum()) <= want.numel() * 1e-4
        assert bool((far <= 2.0 ** -7 * want.float().abs() + 2.0 ** -20 * group).all())


def test_which_gradients_share_a_launch():
    """Fewer tiles than CUs, other Hadamard blocks, extents that the kernel does not serve: two launches, as before."""
    from quartet_amd import _lib
    pairs = _lib.lib().qm_linear_backward_in_one_launch
    assert pairs(4096, 2048, 4096, 32, 32, _lib.QM_BF16, 0) == 1
    assert pairs(9216, 512, 9216, 32, 32, _lib.QM_BF16, 0) == 0      # 144 tiles
    assert pairs(4096, 2080, 4096, 32, 32, _lib.QM_BF16, 0) == 0     # in_features not a multiple of 64
    assert pairs(4096, 2048, 4096, 32, 32, _lib.QM_F32, 3) == 0      # no rotation at all
    assert pairs(0, 2048, 4096, 32, 32, _lib.QM_BF16, 0) == 0 and pairs(4096, 2048, 4100, 32, 32, _lib.QM_BF16, 0) == 0
    assert pairs(4096, 2048, 4096, 48, 32, _lib.QM_BF16, 0) == 0 and pairs(4096, 2048, 4096, 32, 32, 7, 0) == 0
