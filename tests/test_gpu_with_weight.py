"""Producers whose grid quantizes the layer's weight along: both packed operands, bit for bit, as two launches leave them."""
import ctypes

import pytest
import torch

from tests.util import make_input

pytestmark = pytest.mark.gpu


def same_operand(L, a, b, rows, cols):
    """Codes with their padding columns, scales and clip mask of a packed [rows, cols] buffer; the padding rows are nobody's."""
    off = (ctypes.c_size_t * 3)()
    assert L.qm_packed_operand_offsets(rows, cols, off) == 0
    p = (cols + 127) // 128 * 128

    def parts(t):
        codes = t[off[0]: off[0] + (rows + 15) // 16 * 16 * p // 2].view((rows + 15) // 16, p // 128, 16, 64).permute(0, 2, 1, 3).reshape(-1, p // 2)[:rows]
        groups = t[off[1]: off[1] + rows * p // 32].view(rows, p // 32)
        return codes, groups, t[off[2]: off[2] + rows * cols // 8]
    return all(torch.equal(x, y) for x, y in zip(parts(a), parts(b)))


# rows of 16, 32 and 64 lanes; ragged rows and columns of either operand; a weight of fewer and of more workgroups than the rows
@pytest.mark.parametrize("rows,cols,O", [(32, 96, 40), (33, 512, 2056), (70, 640, 1920), (17, 1024, 8), (64, 1728, 640), (40, 4096, 1000)])
@pytest.mark.parametrize("kind", ["norm", "norm+add", "swiglu"])
def test_producer_with_weight(monkeypatch, rows, cols, O, kind):
    print(f"case {kind} with weight {rows}x{cols} {O}", flush=True)
    from quartet_amd import _lib, kernels as K
    L, dev = _lib.lib(), "cuda:0"
    monkeypatch.setattr(K, "_layout", lambda tiled: 2)   # padded
    w = make_input(O, cols, torch.float32, seed=3, scale=0.02).to(dev)
    x = make_input(rows, cols * (2 if kind == "swiglu" else 1), torch.bfloat16 if kind == "swiglu" else torch.float32, seed=4).to(dev)
    add = make_input(rows, cols, torch.bfloat16, seed=5).to(dev) if kind == "norm+add" else None
    gain = (1 + 0.1 * torch.randn(cols, generator=torch.Generator().manual_seed(1))).to(dev)
    signs, signs_w = 0x9E3779B9, 0x0F0F1234
    _, _, want_w = K.linear_forward(make_input(32, cols, torch.float32, seed=6).to(dev), w, 32, None, 32, signs_w, torch.bfloat16, True)
    got, got_w = K.packed_operand_buffer(rows, cols, dev), K.packed_operand_buffer(O, cols, dev)
    tail = (w.data_ptr(), O, K.sign_words(signs_w), got_w.data_ptr(), got_w.numel(), None)
    if kind == "swiglu":
        want = K.swiglu_quantize(x, signs, True)
        rc = L.qm_swiglu_quantize_with_weight_mxfp4(x.data_ptr(), 0, rows, cols, K.sign_words(signs), got.data_ptr(), got.numel(), *tail)
    else:
        want, factor, *total = K.rmsnorm_quantize(x, gain, 1e-5, signs, True, add=add)
        got_factor, got_total = torch.empty_like(factor), torch.empty_like(x)
        rc = L.qm_rmsnorm_quantize_with_weight_mxfp4(x.data_ptr(), 1, add.data_ptr() if add is not None else None, 0, got_total.data_ptr() if add is not None else None,
                                                     gain.data_ptr(), 1e-5, rows, cols, K.sign_words(signs), got.data_ptr(), got.numel(), got_factor.data_ptr(), *tail)
    _lib.check(rc, kind)
    torch.cuda.synchronize()
    assert same_operand(L, got, want, rows, cols) and same_operand(L, got_w, want_w, O, cols)
    if kind != "swiglu":
        assert torch.equal(got_factor, factor) and (add is None or torch.equal(got_total, total[0]))


def test_what_a_producer_with_weight_refuses():
    from quartet_amd import _lib
    L = _lib.lib()
    b = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda:0")
    p, n = b.data_ptr(), b.numel()
    norm = lambda x_dtype=1, add=None, add_dtype=0, rows=16, w=p, O=16, size=n: L.qm_rmsnorm_quantize_with_weight_mxfp4(p, x_dtype, add, add_dtype, p, p, 1e-5, rows, 128, None, p, n, p, w, O, None, p, size, None)
    assert norm(x_dtype=0) == -1 and norm(add=p, add_dtype=1) == -1 and norm(rows=0) == -1 and norm(w=None) == -1 and norm(w=p + 4) == -1 and norm(O=0) == -1 and norm(size=16) == -1
    swiglu = lambda dtype=0, w=p, rows=16: L.qm_swiglu_quantize_with_weight_mxfp4(p, dtype, rows, 128, None, p, n, w, 16, None, p, n, None)
    assert swiglu(dtype=1) == -1 and swiglu(w=None) == -1 and swiglu(rows=0) == -1
