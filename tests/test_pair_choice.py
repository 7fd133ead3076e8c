"""Whether a layer's two gradient products share a launch, asked of the library (no kernel runs)."""
import pytest

from quartet_amd import _lib

WIDTHS = [640, 1024, 1536, 1728, 2048, 3456, 4096, 5504, 8192]


def paths(T, I, O, hd=32):
    """of (gx rotated back by its product, left rotated) x (bf16, fp32 weight gradient)"""
    pairs = _lib.lib().qm_linear_backward_in_one_launch
    return [[pairs(T, I, O, hd, hd, dtype, flags) for dtype in (_lib.QM_BF16, _lib.QM_F32)] for flags in (0, 1)]


@pytest.mark.parametrize("T", [512, 1024, 4096, 8192, 16480, 32768])
def test_a_fused_layer_launches_what_the_unfused_one_does(T):
    """A gradient left rotated for the fused kernel behind it: the weight gradient comes from the same launch, so with the same bits."""
    for I in WIDTHS:
        for O in WIDTHS:
            unfused, fused = paths(T, I, O)
            assert unfused == fused, (T, I, O)


# shapes with a weight gradient (or, few tokens, an input gradient) that launched by itself is cut into K ranges, near the line between one
# launch and two
@pytest.mark.parametrize("T,I,O", [(8192, 1024, 640), (16384, 1536, 1024), (16384, 5504, 512), (16480, 1024, 1536), (16480, 1728, 640), (16480, 1728, 1536),
                                   (32768, 640, 3456), (32768, 1024, 6144), (32768, 2048, 3456), (32768, 4608, 640), (32768, 8192, 640)])
def test_a_cut_product_is_cut_in_every_form(T, I, O):
    """K ranges round differently from whole contractions: one answer for all forms, whatever the weight's type."""
    unfused, fused = paths(T, I, O)
    assert len(set(unfused + fused)) == 1, (unfused, fused)


# steps that measured slower in one launch than in two, for each margin of the choice: kernels of two sorts apart, a cut product, four K steps
# beside long ones, a few long tiles beside tiles of 27 and 32 steps
@pytest.mark.parametrize("T,I,O", [(4096, 4096, 4608), (4096, 2048, 5504), (24576, 6144, 1152), (24576, 11008, 512),
                                   (24576, 8192, 512), (32768, 640, 3456), (24576, 640, 4096)])
def test_two_launches_where_they_are_faster(T, I, O):
    assert [form[0] for form in paths(T, I, O)] == [0, 0]


# and faster in one
@pytest.mark.parametrize("T,I,O,path", [(8192, 4096, 4096, 1), (16384, 4096, 4096, 1), (16480, 3456, 2048, 1), (12288, 7168, 1152, 1), (16384, 1728, 4096, 1),
                                        (32768, 2048, 3072, 1), (16480, 1728, 640, 2), (24576, 4608, 640, 2), (12288, 1152, 1536, 2), (16480, 3456, 512, 2), (512, 640, 1920, 2)])
def test_one_launch_where_it_is_faster(T, I, O, path):
    assert [form[0] for form in paths(T, I, O)] == [path, path]
