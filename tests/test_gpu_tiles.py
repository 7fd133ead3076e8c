"""The product on every tile size and the whole layer on padded operands, at the extents where tiles and padding can go
wrong: below one tile, one row or column past a tile, contractions of one step and of half a step, token counts and widths
that are multiples of 32 only, Hadamard blocks of 32, 64 and 128.  Everything against the oracle."""
import random

import numpy as np
import pytest
import torch

from tests.util import make_input, to_oracle

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("M,N,K", [(1, 8, 128), (33, 72, 384), (64, 32, 128), (65, 64, 640), (130, 264, 640), (300, 384, 1792),   # 64-row tiles
                                   (1000, 520, 256), (513, 1096, 1152), (1025, 2056, 128),                                       # larger tiles
                                   (1063, 576, 1024), (2049, 1024, 1664),                                                        # persistent, ragged rows
                                   (64, 640, 192), (300, 264, 1728)])                                                            # half steps
def test_product_on_ragged_extents(oracle, M, N, K):
    """Row-major operands of any M and N % 8 == 0: fp32 result within accumulation order of the oracle's float64 sums, bf16
    result the rounding of the fp32 one bit for bit (the same sums in the same order)."""
    print(f"case product {M}x{N}x{K}", flush=True)
    from quartet_amd import kernels as Kn
    g = torch.Generator().manual_seed(M + N + K)
    mk = lambda r: (torch.randint(0, 256, (r, K // 2), generator=g, dtype=torch.uint8),
                    torch.randint(120, 131, (r, K // 32), generator=g, dtype=torch.uint8))
    (ac, as_), (bc, bs) = mk(M), mk(N)
    dev = [t.to("cuda:0") for t in (ac, as_, bc, bs)]
    c32 = Kn.gemm_mxfp4_tn(*dev, 1.5, torch.float32, split_k=False)
    c16 = Kn.gemm_mxfp4_tn(*dev, 1.5, torch.bfloat16, split_k=False)
    want = 1.5 * oracle.gemm_tn(ac.numpy(), as_.numpy(), bc.numpy(), bs.numpy())
    assert rel(c32.cpu().numpy(), want) < 1e-5
    assert torch.equal(c16, c32.to(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", [(1, 8, 5376), (33, 72, 4736), (257, 520, 16512), (640, 264, 8256), (1536, 512, 16384)])
def test_product_cut_into_k_ranges(oracle, M, N, K):
    """Few tiles and a long contraction: ranges of unequal length, a last range that ends in half a step.  The same sums in
    another order, each of at most K + ranges fp32 additions (relative error below 1e-5 of the norm); bf16 is the rounding of
    the fp32 result."""
    print(f"case ranges {M}x{N}x{K}", flush=True)
    from quartet_amd import kernels as Kn
    g = torch.Generator().manual_seed(M + N + K)
    mk = lambda r: (torch.randint(0, 256, (r, K // 2), generator=g, dtype=torch.uint8),
                    torch.randint(120, 131, (r, K // 32), generator=g, dtype=torch.uint8))
    (ac, as_), (bc, bs) = mk(M), mk(N)
    dev = [t.to("cuda:0") for t in (ac, as_, bc, bs)]
    c32 = Kn.gemm_mxfp4_tn(*dev, 1.5, torch.float32)
    c16 = Kn.gemm_mxfp4_tn(*dev, 1.5, torch.bfloat16)
    want = 1.5 * oracle.gemm_tn(ac.numpy(), as_.numpy(), bc.numpy(), bs.numpy())
    assert rel(c32.cpu().numpy(), want) < 1e-5
    assert torch.equal(c16, c32.to(torch.bfloat16))


@pytest.mark.parametrize("T,I,O", [(1, 32, 8), (7, 96, 24), (16, 1152, 40), (9, 8192, 264), (16, 10976, 520),   # up to 16 rows: fewer steps than waves, eight waves
                                   (17, 416, 4088), (32, 2048, 4104), (32, 2176, 4104),                          # 32 rows: one workgroup per CU, a short K beyond
                                   (33, 640, 1016), (64, 1664, 4096), (64, 640, 4104), (65, 640, 72)])           # 64 rows, and past every bound
def test_product_of_few_rows(oracle, T, I, O):
    """The layer's forward product at the edges of the kernel for few tokens, against the oracle's float64 sums of the same packed
    operands: fp32 output within K additions (1e-5 of the norm), bf16 output within one rounding of each value (2^-8)."""
    print(f"case few rows T={T} I={I} O={O}", flush=True)
    import quartet_amd as q
    x = make_input(T, I, torch.bfloat16, seed=1, outlier_frac=0.01)
    w = make_input(O, I, torch.bfloat16, seed=2, outlier_frac=0, scale=0.02)
    layer = q.QuantizedLinear(I, O, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(), activation_quantizer=q.QuestMXFP4Quantizer(),
                              gradient_quantizer=q.AlbertTsengQuantizer(), backward_scheme=q.BACKWARD_SCHEMES["Q(E)Q(Wt)t_Q(Et)Q(Xt)t"]())
    layer = layer.to("cuda:0", torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(w.to("cuda:0"))
        y16, y32 = layer(x.to("cuda:0")), layer(x.to("cuda:0").float())
    o = oracle
    qx, qf, qw = (o.quantize(to_oracle(t), 32, mode=o.QUEST_RTN) for t in (x, x.float(), w))
    want, want32 = (o.gemm_tn(a["codes"], a["scales"], qw["codes"], qw["scales"]) for a in (qx, qf))
    assert rel(y32.cpu().numpy(), want32) < 1e-5
    assert rel(y16.float().cpu().numpy(), want) < 2 ** -8


@pytest.mark.parametrize("T,I,O,one_launch", [(1, 32, 8, True), (3, 96, 24, True), (8, 4096, 4096, True), (16, 2048, 520, True), (16, 2080, 520, False), (1, 8160, 264, True),
                                              (2, 16384, 40, True), (1, 1312, 11008, True), (9, 4096, 4096, False), (17, 64, 64, False)])
def test_decode_in_one_launch_is_the_same_layer(T, I, O, one_launch):
    """A few tokens against a packed weight that is kept: quantizer and product in one launch give what the two launches give, bit
    for bit, at the bounds of that kernel (tokens, groups per CU, padded columns, four and eight waves), for both types of x and y
    and with column signs."""
    print(f"case decode T={T} I={I} O={O}", flush=True)
    import quartet_amd as q
    from quartet_amd import _lib
    assert bool(_lib.lib().qm_linear_decode_serves(T, I, O)) == one_launch
    x = make_input(T, I, torch.bfloat16, seed=1, outlier_frac=0.01).to("cuda:0")
    w = make_input(O, I, torch.bfloat16, seed=2, outlier_frac=0, scale=0.02)
    layer = q.QuantizedLinear(I, O, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(), activation_quantizer=q.QuestMXFP4Quantizer(),
                              gradient_quantizer=q.AlbertTsengQuantizer(), backward_scheme=q.BACKWARD_SCHEMES["Q(E)Q(Wt)t_Q(Et)Q(Xt)t"]())
    layer = layer.to("cuda:0", torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(w.to("cuda:0"))
    for signs in (0, 0x9e3779b9):
        layer.activation_quantizer.sign_bits = layer.weight_quantizer.sign_bits = signs
        for xt, amp in ((x, False), (x.float(), False), (x.float(), True)):
            with torch.no_grad(), torch.autocast("cuda", torch.bfloat16, enabled=amp):
                q.enable_packed_weight_cache(layer, False)
                want = layer(xt)
                q.enable_packed_weight_cache(layer)
                layer(xt)                       # fills the cache
                got = layer(xt)
                assert layer.packed_weight_cache.hits == 1
                assert got.dtype == want.dtype and got.shape == want.shape and torch.equal(got, want)
                assert torch.equal(layer(xt[None, :, :])[0], want)


# (T, I, O): K steps from fewer than a request's four to several rounds of eight a wave, with remainders of every kind at a wave's and at a row's end; a tile's
# rows and columns past the end, for tiles of 16 x 16, 32 x 16, 32 x 32, 16 x 64 and 32 x 64; on both sides of the bounds of the kernel
@pytest.mark.parametrize("T,I,O", [(3, 64, 24), (20, 352, 40), (40, 384, 24), (5, 640, 8), (16, 1056, 200), (33, 2176, 40), (24, 4480, 72), (64, 4736, 136), (16, 8960, 24),
                                   (9, 12416, 40), (40, 6400, 56), (17, 8448, 4104), (33, 1152, 4088), (49, 1184, 4104), (64, 1664, 8184), (64, 128, 8200), (31, 2304, 12264),
                                   (32, 2304, 12296), (15, 1152, 11000), (30, 672, 20008)])
def test_product_of_few_rows_with_scales_apart(oracle, T, I, O):
    """The layer's forward product of few tokens where neighbouring groups' scales are up to 2^12 apart, so that a scale taken from another K step shows
    (one group of 400 too large or too small by a factor of two: 10^-2 of the norm and more).  fp32 output against the oracle's float64 sums of the same
    packed operands, within K additions (1e-5 of the norm)."""
    print(f"case few rows, scales apart T={T} I={I} O={O}", flush=True)
    import quartet_amd as q
    g = torch.Generator().manual_seed(T + I + O)
    apart = lambda r: torch.exp2(torch.randint(-3, 4, (r, I // 32), generator=g).float()).repeat_interleave(32, 1)
    x = make_input(T, I, torch.bfloat16, seed=1, outlier_frac=0).float() * apart(T)
    w = (make_input(O, I, torch.bfloat16, seed=2, outlier_frac=0, scale=0.02).float() * apart(O)).to(torch.bfloat16)
    layer = q.QuantizedLinear(I, O, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(), activation_quantizer=q.QuestMXFP4Quantizer(),
                              gradient_quantizer=q.AlbertTsengQuantizer(), backward_scheme=q.BACKWARD_SCHEMES["Q(E)Q(Wt)t_Q(Et)Q(Xt)t"]()).to("cuda:0", torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(w.to("cuda:0"))
        y = layer(x.to("cuda:0"))
    qx, qw = (oracle.quantize(to_oracle(t), 32, mode=oracle.QUEST_RTN) for t in (x, w))
    want = oracle.gemm_tn(qx["codes"], qx["scales"], qw["codes"], qw["scales"])
    assert y.dtype == torch.float32 and rel(y.cpu().numpy(), want) < 1e-5


# groups between the multiplying waves' lanes and sixteen waves' (320, 432, 1020 of them), behind four and eight multiplying waves
@pytest.mark.parametrize("T,I,O", [(5, 2048, 264), (9, 1536, 40), (15, 2176, 520), (2, 9216, 24)])
def test_decode_with_quantizing_waves_beside_the_multiplying_ones(T, I, O):
    test_decode_in_one_launch_is_the_same_layer(T, I, O, True)


# 128 x 128 tiles, at most one to a CU: whole and short last blocks of four K steps (5, 6, 9, 12, 17, 20 steps), one row or eight columns past a tile, 256 of them
@pytest.mark.parametrize("T,I,O", [(641, 1056, 4104), (1000, 2560, 2560), (1537, 1504, 1544), (1025, 640, 3336), (2047, 2176, 1992), (900, 704, 4096)])
def test_products_on_one_large_tile_to_a_cu(T, I, O):
    """A frozen layer's output, whole and by 100 rows (smaller tiles, the same order of additions), in bf16 and in fp32: the same bits."""
    print(f"case one tile to a CU {T}x{I}x{O}", flush=True)
    import quartet_amd as q
    from quartet_amd import _lib
    kernel = lambda rows, dtype: _lib.lib().qm_diag_forward_kernel(rows, I, O, dtype)
    assert kernel(T, _lib.QM_BF16) == kernel(T, _lib.QM_F32) == 32 and kernel(100, _lib.QM_BF16) != 32 and kernel(100, _lib.QM_F32) != 32
    layer = q.QuantizedLinear(I, O, bias=False, device="cuda", dtype=torch.bfloat16, weight_quantizer=q.QuestMXFP4Quantizer(), activation_quantizer=q.QuestMXFP4Quantizer(),
                              gradient_quantizer=q.AlbertTsengQuantizer(), backward_scheme=q.BACKWARD_SCHEMES["Q(E)Q(Wt)t_Q(Et)Q(Xt)t"]())
    with torch.no_grad():
        layer.weight.copy_(make_input(O, I, torch.bfloat16, 1, scale=0.02).cuda())
        x = make_input(T, I, torch.bfloat16, 2).cuda()
        for xt in (x, x.float()):
            whole = layer(xt)
            assert whole.dtype == xt.dtype and torch.isfinite(whole).all()
            for at in range(0, T - 100, 100):
                rows = slice(at, at + 100 if at + 200 <= T else T)
                assert torch.equal(whole[rows], layer(xt[rows].contiguous()))


# workgroups of two, three and four times 16 columns, of which the last one has one, none past the end, or a partial one; more than one to a CU; eight waves to K
@pytest.mark.parametrize("T,I,O", [(16, 640, 4104), (16, 2048, 8192), (9, 1152, 8200), (16, 2048, 8216), (8, 4096, 11008), (5, 96, 12296), (16, 1024, 16408), (4, 8192, 4104), (1, 8320, 8232)])
def test_decode_of_wide_layers(T, I, O):
    test_decode_in_one_launch_is_the_same_layer(T, I, O, True)


@pytest.mark.parametrize("T,I,O,hd", [(32, 32, 32, 32), (4128, 96, 160, 32), (4160, 192, 128, 64), (4224, 128, 256, 128), (96, 160, 96, 32), (288, 192, 320, 32), (544, 1728, 352, 32), (1056, 640, 1088, 32),
                                      (64, 64, 64, 64), (192, 320, 128, 64), (128, 128, 128, 128), (384, 256, 640, 128), (1280, 384, 896, 128)])
def test_layer_on_padded_operands(oracle, T, I, O, hd):
    """Forward and backward of the production layer against the oracle pipeline (same seeds and signs).  bf16 results: each
    stored tensor adds one rounding of relative size 2^-9."""
    print(f"case padded layer T={T} I={I} O={O} hd={hd}", flush=True)
    import quartet_amd as q
    x = make_input(T, I, torch.bfloat16, seed=1, outlier_frac=0.01)
    w = make_input(O, I, torch.bfloat16, seed=2, outlier_frac=0, scale=0.02)
    dy = make_input(T, O, torch.bfloat16, seed=3, outlier_frac=0, scale=1e-3)
    layer = q.QuantizedLinear(I, O, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(hadamard_dim=hd),
                              activation_quantizer=q.QuestMXFP4Quantizer(hadamard_dim=hd),
                              gradient_quantizer=q.AlbertTsengQuantizer(hadamard_dim=hd, stochastic=True, rerotate="signs"),
                              backward_scheme=q.BACKWARD_SCHEMES["Q(E)Q(Wt)t_Q(Et)Q(Xt)t"]()).to("cuda:0", torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(w.to("cuda:0"))
    xd = x.to("cuda:0").requires_grad_(True)
    torch.manual_seed(5)
    random.seed(5)
    y = layer(xd)
    y.backward(dy.to("cuda:0"))
    torch.cuda.synchronize()

    torch.manual_seed(5)
    random.seed(5)
    o = oracle
    signs = np.where(torch.randint(0, 2, (hd,)).numpy() == 0, -1, 1)
    seeds = [random.getrandbits(63) for _ in range(4)]
    d = float(o.FOUR_THIRDS)
    qx = o.quantize(to_oracle(x), hd, mode=o.QUEST_RTN, want_mask=True)
    qw = o.quantize(to_oracle(w), hd, mode=o.QUEST_RTN, want_mask=True)
    y_ref = o.gemm_tn(qx["codes"], qx["scales"], qw["codes"], qw["scales"])
    qe = o.quantize(to_oracle(dy), hd, signs=signs, mode=o.ABSMAX_SR, seed=seeds[0])
    qwt = o.requantize_transposed(qw["codes"], qw["scales"], hd=hd, signs=signs, mode=o.ABSMAX_SR, seed=seeds[1])
    gxq = o.gemm_tn(qe["codes"], qe["scales"], qwt["codes"], qwt["scales"], a_post=d, b_post=d)
    qet = o.quantize(to_oracle(dy), hd, signs=signs, mode=o.ABSMAX_SR, transposed_in=True, seed=seeds[2])
    qxt = o.requantize_transposed(qx["codes"], qx["scales"], hd=hd, signs=signs, mode=o.ABSMAX_SR, seed=seeds[3])
    gwq = o.gemm_tn(qet["codes"], qet["scales"], qxt["codes"], qxt["scales"], a_post=d, b_post=d)
    ste = lambda g, qd: o.masked_hadamard_bwd(g.astype(np.float32), hd, o.BF16, None, qd["mask"], out_dtype=o.F32)
    assert rel(y.detach().float().cpu().numpy(), y_ref) <= 3e-3
    assert rel(xd.grad.float().cpu().numpy(), ste(gxq, qx)) <= 5e-3
    assert rel(layer.weight.grad.float().cpu().numpy(), ste(gwq, qw)) <= 5e-3


def error_only_layer(q, I, O, hd, dtype):
    return q.QuantizedLinear(I, O, bias=False, weight_quantizer=q.QuestMXFP4Quantizer(hadamard_dim=hd),
                             activation_quantizer=q.QuestMXFP4Quantizer(hadamard_dim=hd),
                             gradient_quantizer=q.AlbertTsengQuantizer(hadamard_dim=hd, stochastic=True),
                             backward_scheme=q.BACKWARD_SCHEMES["Q(E)W_Q(Et)X"]()).to("cuda:0", dtype)


@pytest.mark.parametrize("T,I,O,hd,wide,spread",
                         [(*case, s) for case in [(32, 32, 32, 32, False), (96, 160, 1056, 32, True), (256, 384, 640, 128, False)] for s in (0, 26, 28, 29, 60)] +
                         [(544, 1728, 352, 32, False, 0), (4160, 192, 128, 64, True, 28), (4160, 192, 128, 64, True, 29), (1152, 2048, 2176, 32, False, 28)])
def test_error_only_layer_on_packed_operands(oracle, monkeypatch, T, I, O, hd, wide, spread):
    """Scheme Q(E)W_Q(Et)X on packed operands, widened to eight bits for its products, against the oracle's de-quantized
    tensors multiplied in float64.  spread: all but every seventh row of x and of W are scaled by 2^spread, so that the row scales
    of a block of 32 lie within the eight-bit format (28 octaves) or not.  bf16 results: one rounding of the product and one of the
    rotation, each of relative size 2^-9, against the oracle's bf16 product rotated exactly."""
    print(f"case error-only T={T} I={I} O={O} hd={hd} wide={wide} spread={spread}", flush=True)
    import quartet_amd as q
    from quartet_amd import kernels as Kn
    monkeypatch.setattr(Kn, "gemm_mxfp4_bf16_nn", lambda *a, **k: pytest.fail("left the packed path"))
    scaled = lambda t: torch.where(torch.arange(t.shape[0]).unsqueeze(1) % 7 == 3, t.float(), t.float() * 2.0 ** spread).to(t.dtype)
    x = scaled(make_input(T, I, torch.bfloat16, seed=1, outlier_frac=0.01))
    w = scaled(make_input(O, I, torch.bfloat16, seed=2, outlier_frac=0, scale=0.02))
    idx = np.arange(hd)
    parity = np.array([[bin(i & j).count("1") & 1 for j in idx] for i in idx])
    if spread:
        # an error signal that, rotated along either axis, is nonzero only where the other operand's row is a small one, so that
        # nothing larger hides what is lost: whole numbers, which neither bf16 nor the rotation rounds
        pick = torch.Generator().manual_seed(4)
        s = torch.randint(0, 2, (T, O), generator=pick).double() * 2 - 1
        s *= (torch.arange(T) % 7 == 3).unsqueeze(1) * (torch.arange(O) % 7 == 3)
        sign = torch.from_numpy(np.where(parity, -1.0, 1.0))
        s = (s.view(-1, hd) @ sign).view(T, O)
        e = ((s.T.reshape(-1, hd) @ sign).view(O, T).T * 2.0 ** -10).to(torch.bfloat16).contiguous()
    else:
        e = make_input(T, O, torch.bfloat16, seed=3, outlier_frac=0, scale=1e-3)
    layer = error_only_layer(q, I, O, hd, torch.float32 if wide else torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(w.to("cuda:0"))
    xd = x.to("cuda:0").requires_grad_(True)
    random.seed(5)
    with torch.autocast("cuda", torch.bfloat16, enabled=wide):
        y = layer(xd)
        y.backward(e.to("cuda:0"))
    torch.cuda.synchronize()
    random.seed(5)
    o, d = oracle, float(oracle.FOUR_THIRDS)
    qx = o.quantize(to_oracle(x), hd, mode=o.QUEST_RTN, want_mask=True)
    qw = o.quantize(to_oracle(w.float() if wide else w), hd, mode=o.QUEST_RTN, want_mask=True)
    qe = o.quantize(to_oracle(e), hd, mode=o.ABSMAX_SR, seed=random.getrandbits(63))
    qet = o.quantize(to_oracle(e), hd, mode=o.ABSMAX_SR, transposed_in=True, seed=random.getrandbits(63))
    xv, wv = o.dequantize(qx["codes"], qx["scales"], 1.0).astype(np.float64), o.dequantize(qw["codes"], qw["scales"], 1.0).astype(np.float64)
    ev, etv = o.dequantize(qe["codes"], qe["scales"], d).astype(np.float64), o.dequantize(qet["codes"], qet["scales"], d).astype(np.float64)
    c = float(torch.tensor(hd ** -0.5).to(torch.bfloat16))
    H = np.where(parity, -c, c)

    def rotate(p, mask):
        keep = np.unpackbits(np.asarray(mask).reshape(p.shape[0], -1), axis=1, bitorder="little")
        return ((torch.from_numpy(p).to(torch.bfloat16).double().numpy() * keep).reshape(-1, hd) @ H.T).reshape(p.shape)
    assert rel(y.detach().float().cpu(), xv @ wv.T) < 4e-3
    assert rel(xd.grad.float().cpu(), rotate(ev @ wv, qx["mask"])) < 4e-3
    assert rel(layer.weight.grad.float().cpu(), rotate(etv @ xv, qw["mask"])) < 4e-3


# contractions of 4, 6, 7, 8, 10, 11, 12 and 33 steps of 128: whole and short last blocks of four steps.  From 4, 8, 11, 12, ... steps
# on, blocks of 512 rows and 256 columns whose row scales lie within five octaves are widened to six bits, others to eight.
@pytest.mark.parametrize("T,I,O,spread", [(512, 192, 768, 0), (896, 256, 1024, 0), (1280, 320, 1408, 0), (1536, 2048, 896, 0)] +
                         [(*case, s) for case in [(512, 320, 512), (1536, 96, 1408), (4224, 544, 640)] for s in (4, 5, 6, 12)])
def test_error_only_layer_on_whole_steps(oracle, monkeypatch, T, I, O, spread):
    test_error_only_layer_on_packed_operands(oracle, monkeypatch, T, I, O, 32, True, spread)


@pytest.mark.parametrize("T,I,O", [(4224, 544, 1408), (2048, 2048, 4096)])
def test_error_only_layer_with_both_widths_in_one_product(oracle, T, I, O):
    """Outliers in single blocks of 512 rows and 256 columns, the last block among them, zero rows (which count for no range) and
    rows as small as a zero group's scale: every column group of 32 against float64, with the tolerance of the test above."""
    print(f"case error-only widths T={T} I={I} O={O}", flush=True)
    import quartet_amd as q
    x = make_input(T, I, torch.bfloat16, seed=1, outlier_frac=0).float()
    w = make_input(O, I, torch.bfloat16, seed=2, outlier_frac=0, scale=0.02).float()
    x[600:640, 256:300] *= 2.0 ** 7
    x[T - 20:, :32] *= 2.0 ** 9
    x[1030:1040] = 0.0
    x[1100:1110, 64:96] *= 2.0 ** -24
    x[1600:1610, I - 32:] *= 2.0 ** -28
    w[O - 3, 300:320] *= 2.0 ** 8
    x, w = x.to(torch.bfloat16), w.to(torch.bfloat16)
    e = make_input(T, O, torch.bfloat16, seed=3, outlier_frac=0, scale=1e-3)
    layer = error_only_layer(q, I, O, 32, torch.bfloat16)
    with torch.no_grad():
        layer.weight.copy_(w.to("cuda:0"))
    xd = x.to("cuda:0").requires_grad_(True)
    random.seed(5)
    layer(xd).backward(e.to("cuda:0"))
    torch.cuda.synchronize()
    random.seed(5)
    o, d = oracle, float(oracle.FOUR_THIRDS)
    qx, qw = (o.quantize(to_oracle(t), 32, mode=o.QUEST_RTN, want_mask=True) for t in (x, w))
    qe = o.quantize(to_oracle(e), 32, mode=o.ABSMAX_SR, seed=random.getrandbits(63))
    qet = o.quantize(to_oracle(e), 32, mode=o.ABSMAX_SR, transposed_in=True, seed=random.getrandbits(63))
    on_gpu = lambda t, scale: torch.from_numpy(o.dequantize(t["codes"], t["scales"], scale)).to("cuda:0").double()
    parity = torch.tensor([[bin(i & j).count("1") & 1 for j in range(32)] for i in range(32)], device="cuda:0")
    H = torch.where(parity == 1, -1.0, 1.0).double() * float(torch.tensor(32 ** -0.5).to(torch.bfloat16))

    def groups(p, mask):   # the bf16 product, masked and rotated, as groups of 32 columns
        keep = torch.from_numpy(np.unpackbits(np.asarray(mask).reshape(p.shape[0], -1), axis=1, bitorder="little")).to("cuda:0")
        return (p.to(torch.bfloat16).double() * keep).view(p.shape[0], -1, 32) @ H
    for got, want in [(xd.grad, groups(on_gpu(qe, d) @ on_gpu(qw, 1.0), qx["mask"])),
                      (layer.weight.grad, groups(on_gpu(qet, d) @ on_gpu(qx, 1.0), qw["mask"]))]:
        err = (got.double().view(want.shape) - want).square().sum((0, 2)).sqrt() / want.square().sum((0, 2)).sqrt()
        assert float(err.max()) < 4e-3, float(err.max())
