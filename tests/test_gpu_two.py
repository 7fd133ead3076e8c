"""The product on 256 x 192 tiles, two workgroups to a CU, at the extents where its tiles, K steps and blocks of scales can go wrong.  The
shapes are ones that it is chosen for (more tiles than CUs); the other kernels are reached by smaller slices of the same operands."""
import pytest
import torch

from tests.util import make_input

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,I,O", [(33000, 768, 576),      # three columns of tiles, ragged rows, six steps: a short last block of scales
                                   (4100, 1152, 4104),     # ragged both ways by a piece of eight columns and four rows, nine steps
                                   (8200, 1664, 2056),     # thirteen steps
                                   (8192, 1504, 4608),     # whole tiles, in_features padded to 1536
                                   (131072, 512, 776),     # four steps, several tiles a workgroup
                                   (5793, 2304, 8264)])    # odd rows, eighteen steps, several tiles a workgroup
def test_products_on_two_workgroups_to_a_cu(T, I, O):
    """A frozen layer's output, whole and by 500 rows (another kernel, the same order of additions): the same bits."""
    print(f"case two {T}x{I}x{O}", flush=True)
    import quartet_amd as q
    from quartet_amd import _lib
    kernel = lambda rows: _lib.lib().qm_diag_forward_kernel(rows, I, O, _lib.QM_BF16)
    assert kernel(T) == 3 and kernel(500) != 3
    layer = q.QuantizedLinear(I, O, bias=False, device="cuda", dtype=torch.bfloat16, weight_quantizer=q.QuestMXFP4Quantizer(),
                              activation_quantizer=q.QuestMXFP4Quantizer(), gradient_quantizer=q.AlbertTsengQuantizer(stochastic=True),
                              backward_scheme=q.BACKWARD_SCHEMES["Q(E)Q(Wt)t_Q(Et)Q(Xt)t"]())
    with torch.no_grad():
        layer.weight.copy_(make_input(O, I, torch.bfloat16, 1, scale=0.02).cuda())
        x = make_input(T, I, torch.bfloat16, 2).cuda()
        whole = layer(x)
        assert torch.isfinite(whole).all()
        for rows in (slice(0, 500), slice(T // 2, T // 2 + 500), slice(T - 500, T)):
            assert torch.equal(whole[rows], layer(x[rows].contiguous()))
        # the tokens in between, from several launches of a repeated pass into other memory
        junk = torch.full_like(whole, float("nan"))
        del junk
        assert torch.equal(whole, layer(x))


def test_two_workgroups_against_the_product_in_float64():
    """bf16 of fp32 sums: eight significant bits, so a result is off by 2^-8 of itself at most, with the sums' own rounding (below 1e-5 of the
    largest result of its row, K = 1536 terms) beside it."""
    from quartet_amd import kernels as K
    g = torch.Generator().manual_seed(5)
    M, N, Kd = 8192, 4608, 1536
    assert K._lib.lib().qm_diag_forward_kernel(M, Kd, N, K._lib.QM_BF16) == 3
    mk = lambda r: (torch.randint(0, 256, (r, Kd // 2), generator=g, dtype=torch.uint8).cuda(), torch.randint(124, 129, (r, Kd // 32), generator=g, dtype=torch.uint8).cuda())
    (ac, as_), (bc, bs) = mk(M), mk(N)
    got = K.gemm_mxfp4_tn(K.tile_codes(ac), as_, K.tile_codes(bc), bs, 1.5, a_tiled=True, b_tiled=True)
    rows = torch.tensor([0, 1, 127, 128, 255, 256, 4095, 8191], device="cuda")
    a = K.dequantize_mxfp4(ac[rows].contiguous(), as_[rows].contiguous()).double()
    b = K.dequantize_mxfp4(bc, bs).double()
    want = 1.5 * (a.cpu() @ b.cpu().T)
    err = (got[rows].double().cpu() - want).abs()
    assert (err <= want.abs() * 2.0 ** -8 + 1e-5 * want.abs().amax(dim=1, keepdim=True)).all()
    assert torch.equal(got, K.gemm_mxfp4_tn(ac, as_, bc, bs, 1.5))   # row-major operands: another kernel
