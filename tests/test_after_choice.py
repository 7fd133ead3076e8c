"""Whether an evaluated model's rotary split runs in the epilogue of its projection, asked of the library (no kernel runs)."""
import pytest

from quartet_amd import _lib


# measured: a few hundred tokens are one round of smaller tiles and a short launch behind it; 128 x 128 tiles take longer than both
@pytest.mark.parametrize("T,n_embd", [(65, 640), (256, 640), (65, 1536), (128, 1536), (200, 1280), (128, 2048), (96, 2560), (128, 4096)])
def test_rotary_split_of_few_tokens_is_a_launch_of_its_own(T, n_embd):
    assert _lib.lib().qm_linear_rope_serves(T, n_embd, n_embd, 128 if n_embd % 128 == 0 else 64) == 0


@pytest.mark.parametrize("T,n_embd", [(1024, 640), (512, 1536), (300, 2048), (384, 2560), (256, 4096), (4096, 2560), (4096, 3584), (32768, 1536)])
def test_rotary_split_of_more_tokens_rides_along(T, n_embd):
    assert _lib.lib().qm_linear_rope_serves(T, n_embd, n_embd, 128) == 1


@pytest.mark.parametrize("T,n_embd,hidden", [(65, 640, 1728), (4096, 640, 1728), (32768, 1536, 4096), (300, 4096, 11008)])
def test_swiglu_rides_along(T, n_embd, hidden):
    assert _lib.lib().qm_linear_swiglu_serves(T, n_embd, hidden) == 1
