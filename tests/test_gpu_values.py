"""The quantizer modules' kernel: de-quantized values and clip mask alone, in whole waves and in a last one that is not."""
import numpy as np
import pytest
import torch

from tests.util import from_oracle_bf16, make_input, to_oracle

pytestmark = pytest.mark.gpu


# one chunk, less than a wave, whole waves and workgroups, one group past each
@pytest.mark.parametrize("rows,cols", [(1, 128), (3, 640), (16, 128), (64, 128), (65, 128), (7, 1152), (33, 2048)])
@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", ["QUEST_RTN", "ABSMAX_RTN", "ABSMAX_SR", "QUEST_SR"])
def test_values_are_those_of_the_codes(oracle, rows, cols, hd, dtype, mode):
    """Bit for bit the oracle's values and mask, with column signs, ties, zeros, outliers, and groups at both ends of the exponents."""
    print(f"case values {rows}x{cols} hd={hd} {dtype} {mode}", flush=True)
    from quartet_amd import _lib, kernels as K
    x = make_input(rows, cols, dtype, seed=rows + cols + hd, outlier_frac=0.01)
    x[0, :hd] = 0
    x.view(-1)[-hd:] *= 2.0 ** 115     # scales near the top: values below infinity
    if rows > 2:
        x[1, :hd] *= 2.0 ** -130       # subnormal inputs
        x[2, :hd] = torch.tensor([0.0, -0.0, 1.0, -1.0] * (hd // 4), dtype=dtype)
    signs = (0x9E3779B97F4A7C15F39CC0605CEDC835 >> 3) & ((1 << hd) - 1)
    xd = x.to("cuda:0")
    code, quest = getattr(K, "QM_" + mode), mode.startswith("QUEST")
    values = torch.full_like(xd, float("nan"))
    mask = torch.zeros(rows * cols // 8, dtype=torch.uint8, device="cuda:0")
    rc = _lib.lib().qm_pseudo_quantize_mxfp4(xd.data_ptr(), 0 if dtype == torch.bfloat16 else 1, rows, cols, hd, K.sign_words(signs), code, 77,
                                             mask.data_ptr() if quest else None, values.data_ptr(), None)
    _lib.check(rc, "qm_pseudo_quantize_mxfp4")
    torch.cuda.synchronize()
    sv = np.array([-1 if (signs >> j) & 1 else 1 for j in range(hd)])
    ref = oracle.quantize(to_oracle(x), hd, signs=sv, mode=getattr(oracle, mode), seed=77, want_mask=quest, want_dequant=True)
    want = from_oracle_bf16(ref["dequant"]) if dtype == torch.bfloat16 else torch.from_numpy(ref["dequant"])
    as_int = torch.int16 if dtype == torch.bfloat16 else torch.int32
    assert torch.equal(values.cpu().view(as_int).view(-1), want.contiguous().view(as_int).view(-1))
    if quest:
        assert np.array_equal(mask.cpu().numpy(), ref["mask"].reshape(-1))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hd", [32, 128])
@pytest.mark.parametrize("mode", ["QUEST_RTN", "ABSMAX_RTN", "ABSMAX_SR", "QUEST_SR"])
def test_the_mask_may_be_left_out_or_asked_for(mode, hd, dtype):
    """Either way the values and masks of the quantizer that writes codes, too."""
    from quartet_amd import _lib, kernels as K
    print(f"case values with and without mask hd={hd} {dtype} {mode}", flush=True)
    rows, cols, code = 37, 1152, getattr(K, "QM_" + mode)
    x = make_input(rows, cols, dtype, seed=hd, outlier_frac=0.01).to("cuda:0")
    _, _, want_mask, want = K.quantize_mxfp4(x, hd, 0x5A5A1234, code, seed=77, want_mask=True, want_dequant=True)
    for with_mask in (False, True):
        values, mask = torch.full_like(x, float("nan")), torch.zeros(rows * cols // 8, dtype=torch.uint8, device="cuda:0")
        rc = _lib.lib().qm_pseudo_quantize_mxfp4(x.data_ptr(), _lib.QM_BF16 if dtype == torch.bfloat16 else _lib.QM_F32, rows, cols, hd, K.sign_words(0x5A5A1234), code, 77,
                                                 mask.data_ptr() if with_mask else None, values.data_ptr(), None)
        _lib.check(rc, "qm_pseudo_quantize_mxfp4")
        assert torch.equal(values, want.view(values.shape))
        assert torch.equal(mask, want_mask.view(-1)) if with_mask else not mask.any()


def test_values_of_nothing_and_of_misaligned_tensors():
    from quartet_amd import _lib, kernels as K
    L = _lib.lib()
    x = torch.randn(4, 128, device="cuda:0", dtype=torch.bfloat16)
    y = torch.empty_like(x)
    call = lambda src, dst, rows=4, cols=128, hd=64, mode=0, mask=None: L.qm_pseudo_quantize_mxfp4(src, 0, rows, cols, hd, None, mode, 0, mask, dst, None)
    assert call(x.data_ptr(), y.data_ptr(), rows=0) == 0
    assert call(x.data_ptr() + 2, y.data_ptr()) == -2 and call(x.data_ptr(), y.data_ptr() + 8) == -2
    assert call(None, y.data_ptr()) == -1 and call(x.data_ptr(), None) == -1
    assert call(x.data_ptr(), y.data_ptr(), cols=96) == -1 and call(x.data_ptr(), y.data_ptr(), hd=1) == -1 and call(x.data_ptr(), y.data_ptr(), mode=4) == -1
