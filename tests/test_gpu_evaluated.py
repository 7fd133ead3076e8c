"""Products of an evaluated model whose epilogue goes on with their result, and its last norm."""
import ctypes

import numpy as np
import pytest
import torch

from tests.util import make_input

pytestmark = pytest.mark.gpu
BF16, LAYOUT_PADDED = torch.bfloat16, 2


def packed(K, monkeypatch, x, w):
    """The padded operands of a layer, as its forward pass leaves them, and its bf16 result."""
    monkeypatch.setattr(K, "_layout", lambda tiled: LAYOUT_PADDED)
    y, px, pw = K.linear_forward(x, w, 32, 0x5A5A5A5A, 32, 0x0F0F1234, BF16, True)
    return y, px, pw


def codes_and_scales(K, buffer, rows, cols):
    off = (ctypes.c_size_t * 3)()
    from quartet_amd import _lib
    assert _lib.lib().qm_packed_operand_offsets(rows, cols, off) == 0
    padded = (cols + 127) // 128 * 128
    tiles = buffer[off[0]: off[0] + (rows + 15) // 16 * 16 * padded // 2].view((rows + 15) // 16, padded // 128, 16, 64)
    codes = tiles.permute(0, 2, 1, 3).reshape(-1, padded // 2)[:rows]
    return codes, buffer[off[1]: off[1] + rows * padded // 32].view(rows, padded // 32)


# one tile and several, ragged rows, an odd and an even number of groups, whole tiles of padding behind the columns, fewer K steps than four
@pytest.mark.parametrize("T,I,hidden", [(65, 96, 32), (127, 640, 96), (129, 512, 1696), (384, 544, 1728), (1000, 640, 160), (513, 1536, 4096)])
@pytest.mark.parametrize("signs", [None, 0x9E3779B9])
def test_swiglu_and_quantizer_in_the_product(monkeypatch, T, I, hidden, signs):
    """Codes and scales, padding included, bit for bit those of the product, then the producer."""
    print(f"case product with SwiGLU {T}x{I}x2*{hidden}", flush=True)
    from quartet_amd import _lib, kernels as K
    x = make_input(T, I, BF16, seed=1, outlier_frac=0.01).to("cuda:0")
    w = make_input(2 * hidden, I, BF16, seed=2, outlier_frac=0, scale=0.05).to("cuda:0")
    h12, px, pw = packed(K, monkeypatch, x, w)
    want = codes_and_scales(K, K.swiglu_quantize(h12, signs, True), T, hidden)
    out = K.packed_operand_buffer(T, hidden, x.device).fill_(0xA5)
    rc = _lib.lib().qm_linear_swiglu_quantize(px.data_ptr(), px.numel(), pw.data_ptr(), pw.numel(), T, I, hidden, K.sign_words(signs), out.data_ptr(), out.numel(), None)
    _lib.check(rc, "qm_linear_swiglu_quantize")
    for got, ref in zip(codes_and_scales(K, out, T, hidden), want):
        assert torch.equal(got, ref)


# sequences shorter and longer than a pass over a tile's rows, of one token, rows over the tile's edge; heads narrower than a tile and wider
@pytest.mark.parametrize("B,S,I,heads,hs", [(8, 512, 640, 5, 128), (3, 43, 96, 3, 8), (130, 1, 160, 2, 64), (5, 17, 512, 1, 136), (9, 15, 256, 4, 72)])
def test_rotary_split_in_the_product(monkeypatch, B, S, I, heads, hs):
    print(f"case product with rotary split {B}x{S}x{I} heads={heads}x{hs}", flush=True)
    from quartet_amd import _lib, kernels as K
    from quartet_amd.llama import rotary_table
    T, C = B * S, heads * hs
    x = make_input(T, I, BF16, seed=1, outlier_frac=0.01).to("cuda:0")
    w = make_input(3 * C, I, BF16, seed=2, outlier_frac=0, scale=0.05).to("cuda:0")
    table = rotary_table(hs, S).to("cuda:0").contiguous()
    qkv, px, pw = packed(K, monkeypatch, x, w)
    want = [torch.empty(T, C, dtype=BF16, device="cuda:0") for _ in range(3)]
    got = [torch.full_like(t, float("nan")) for t in want]
    L = _lib.lib()
    _lib.check(L.qm_rope_split_qkv(qkv.data_ptr(), 0, T, S, C, hs, table.data_ptr(), *[t.data_ptr() for t in want], 0, None), "qm_rope_split_qkv")
    rc = L.qm_linear_rope(px.data_ptr(), px.numel(), pw.data_ptr(), pw.numel(), T, I, C, hs, S, table.data_ptr(), *[t.data_ptr() for t in got], None)
    _lib.check(rc, "qm_linear_rope")
    for g, r in zip(got, want):
        assert torch.equal(g, r)


def test_what_those_products_refuse():
    from quartet_amd import _lib
    L = _lib.lib()
    b = torch.empty(1 << 22, dtype=torch.uint8, device="cuda:0")
    p, n = b.data_ptr(), b.numel()
    swiglu = lambda T=128, I=128, hidden=64, px=p, size=n, out=p: L.qm_linear_swiglu_quantize(px, size, p, n, T, I, hidden, None, out, n, None)
    assert swiglu(T=64) == -1 and swiglu(I=100) == -1 and swiglu(hidden=48) == -1 and swiglu(px=None) == -1 and swiglu(size=64) == -1 and swiglu(out=p + 16) == -1
    rope = lambda T=128, I=128, C=64, hs=8, S=16, q=p, table=p: L.qm_linear_rope(p, n, p, n, T, I, C, hs, S, table, q, p, p, None)
    assert rope(T=64) == -1 and rope(hs=12) == -1 and rope(C=60, hs=8) == -1 and rope(S=0) == -1 and rope(q=None) == -1 and rope(table=p + 4) == -1
    assert L.qm_linear_swiglu_serves(64, 640, 1728) == 0 and L.qm_linear_rope_serves(4096, 640, 640, 12) == 0


@pytest.mark.parametrize("add_dtype", [None, BF16, torch.float32])
def test_an_evaluated_model_is_the_same_model(add_dtype):
    """With packed weights kept, without (two launches instead of one), and the residual sum: the same bits; and gradients go on asking
    for the path that keeps what they need."""
    import quartet_amd as q
    from quartet_amd.fused import rmsnorm_rope_linear, rmsnorm_swiglu_linear
    from quartet_amd.llama import Llama, llama_30m, rotary_table
    torch.manual_seed(3)
    with torch.device("cuda"):
        model = Llama(llama_30m(n_layer=1, sequence_length=128)).eval()
    block = model.transformer.h[0]
    x = make_input(288, 640, torch.float32, seed=5).view(3, 96, 640).to("cuda:0")
    add = None if add_dtype is None else make_input(288, 640, add_dtype, seed=6).view(3, 96, 640).to("cuda:0")
    table = rotary_table(128, 96).to("cuda:0")

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16):
            return (*rmsnorm_swiglu_linear(block.ln_2, block.mlp.w12, block.mlp.c_proj, x, add=add),
                    *rmsnorm_rope_linear(block.ln_1, block.attn.c_attn, x, table, 5, add=add))
    want = run()
    q.enable_packed_weight_cache(model)
    run()                                   # quantizes the weights
    got = run()
    assert all(m.packed_weight_cache.hits == 1 for m in (block.mlp.w12, block.mlp.c_proj, block.attn.c_attn))
    for g, r in zip(got, want):
        assert g.dtype == r.dtype and g.shape == r.shape and torch.equal(g, r)
    with torch.no_grad():
        block.mlp.w12.weight.mul_(2.0)      # a kept form that is out of date is not used
        changed = run()[0]
        q.enable_packed_weight_cache(model, False)
    assert torch.equal(changed, run()[0]) and not torch.equal(changed, want[0])
    xg = x.clone().requires_grad_(True)
    q.enable_packed_weight_cache(model)
    for _ in range(2):
        with torch.autocast("cuda", dtype=BF16):
            y, _ = rmsnorm_swiglu_linear(block.ln_2, block.mlp.w12, block.mlp.c_proj, xg, add=add)
        y.float().sum().backward()
    assert torch.isfinite(xg.grad).all() and block.mlp.w12.weight.grad is not None


def test_an_evaluated_attention_of_many_tokens_is_the_same():
    """Enough tokens for the rotary split to ride along: the bits of the two launches."""
    import quartet_amd as q
    from quartet_amd import _lib
    from quartet_amd.fused import rmsnorm_rope_linear
    from quartet_amd.llama import Llama, llama_30m, rotary_table
    torch.manual_seed(3)
    with torch.device("cuda"):
        block = Llama(llama_30m(n_layer=1, sequence_length=512)).eval().transformer.h[0]
    x = make_input(1100, 640, torch.float32, seed=5).view(5, 220, 640).to("cuda:0")
    add = make_input(1100, 640, BF16, seed=6).view(5, 220, 640).to("cuda:0")
    table = rotary_table(128, 220).to("cuda:0")
    assert _lib.lib().qm_linear_rope_serves(1100, 640, 640, 128) == 1

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16):
            return rmsnorm_rope_linear(block.ln_1, block.attn.c_attn, x, table, 5, add=add)
    want = run()
    q.enable_packed_weight_cache(block)
    run()                                   # quantizes the weight
    for g, r in zip(run(), want):
        assert g.dtype == r.dtype and g.shape == r.shape and torch.equal(g, r)


@pytest.mark.parametrize("rows,cols", [(1, 4), (5, 640), (4, 768), (7, 772), (3, 1536), (9, 1540), (2, 4096)])
@pytest.mark.parametrize("add_dtype", [None, BF16, torch.float32])
@pytest.mark.parametrize("out_dtype", [BF16, torch.float32])
def test_last_norm(rows, cols, add_dtype, out_dtype):
    """Against float64: the fp32 sum of at most 16 + 6 additions in a row, a root, a quotient and three products: 2^-24 each, 25 of them;
    bf16 results one rounding to eight significant bits more, 2^-8."""
    from quartet_amd import kernels as K
    x = make_input(rows, cols, torch.float32, seed=rows + cols)
    add = None if add_dtype is None else make_input(rows, cols, add_dtype, seed=3)
    gain = 1 + 0.1 * torch.randn(cols, generator=torch.Generator().manual_seed(1))
    s = (x if add is None else x + add.float()).double()
    want = s / torch.sqrt((s * s).mean(-1, keepdim=True) + 1e-5) * gain.double()
    got = K.rmsnorm(x.to("cuda:0"), gain.to("cuda:0"), 1e-5, None if add is None else add.to("cuda:0"), out_dtype).cpu()
    assert got.dtype == out_dtype
    err = ((got.double() - want).abs() / want.abs().clamp_min(1e-30)).numpy()
    assert np.all(err <= 25 * 2.0 ** -24 + (2.0 ** -8 if out_dtype == BF16 else 0.0))


def test_last_norm_of_more_rows_than_a_grid_holds():
    """64 threads a row and fewer than 2^32 threads in a launch: every row past 2^25 and 2^26 is what it is by itself."""
    from quartet_amd import kernels as K
    rows = (1 << 26) + 5
    print(f"case last norm of {rows} rows", flush=True)
    x = torch.randn(rows, 4, device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(2))
    add = torch.randn(rows, 4, device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(3)).to(BF16)
    gain = torch.tensor([0.5, 1.0, 1.5, 2.0], device="cuda:0")
    got = K.rmsnorm(x, gain, 1e-5, add, BF16)
    for at in (0, (1 << 25) - 4, 1 << 25, (1 << 26) - 4, 1 << 26):
        part = slice(at, at + 9)
        assert torch.equal(got[part], K.rmsnorm(x[part].contiguous(), gain, 1e-5, add[part].contiguous(), BF16))


def test_last_norm_of_a_model_takes_the_module_where_somebody_listens_or_asks_for_gradients():
    from quartet_amd.fused import rmsnorm
    from quartet_amd.llama import RMSNorm
    class Head(torch.nn.Linear):
        pass
    norm, head = RMSNorm(640).to("cuda:0"), torch.nn.Linear(640, 8, bias=False).to("cuda:0")
    x = torch.randn(2, 70, 640, device="cuda:0")
    with torch.autocast("cuda", dtype=BF16):
        with torch.no_grad():
            one = rmsnorm(norm, head, x)
            assert one.dtype == BF16 and float((one.float() - norm(x)).abs().max()) < 2.0 ** -6
            seen = []
            handle = norm.register_forward_hook(lambda *a: seen.append(1))
            assert torch.equal(rmsnorm(norm, head, x), norm(x)) and len(seen) == 2
            handle.remove()
            # another head, or one that somebody watches, sees the norm's own result
            assert rmsnorm(norm, Head(640, 8, device="cuda:0"), x).dtype == torch.float32
            handle = head.register_forward_pre_hook(lambda *a: None)
            assert torch.equal(rmsnorm(norm, head, x), norm(x))
            handle.remove()
        y = rmsnorm(norm, head, x)
        assert y.dtype == torch.float32 and y.requires_grad
    with torch.no_grad():
        assert torch.equal(rmsnorm(norm, head, x, x), norm(x + x))


def test_rows_that_are_not_the_layer_s_are_refused_as_without_packed_weights():
    """An input of twice the layer's width is as many rows again: nothing may be launched for them on results of half the size."""
    import quartet_amd as q
    from quartet_amd.fused import rmsnorm_rope_linear, rmsnorm_swiglu_linear
    from quartet_amd.llama import LlamaBlock, RMSNorm, llama_30m, rotary_table
    with torch.device("cuda"):
        block, wide = LlamaBlock(llama_30m(n_layer=1)).eval(), RMSNorm(1280)
    q.enable_packed_weight_cache(block)
    table = rotary_table(128, 96).to("cuda:0")
    with torch.no_grad(), torch.autocast("cuda", dtype=BF16):
        x = torch.randn(3, 96, 640, device="cuda:0")
        rmsnorm_rope_linear(block.ln_1, block.attn.c_attn, x, table, 5)
        rmsnorm_swiglu_linear(block.ln_2, block.mlp.w12, block.mlp.c_proj, x)
        for norm in (block.ln_1, wide):
            with pytest.raises(RuntimeError):
                rmsnorm_rope_linear(norm, block.attn.c_attn, torch.randn(3, 96, 1280, device="cuda:0"), table, 5)
            with pytest.raises(RuntimeError):
                rmsnorm_swiglu_linear(norm, block.mlp.w12, block.mlp.c_proj, torch.randn(3, 96, 1280, device="cuda:0"))


def _head(T, K, V, add_dtype, seed):
    from quartet_amd.llama import RMSNorm
    norm, head = RMSNorm(K).to("cuda:0"), torch.nn.Linear(K, V, bias=False).to("cuda:0")
    g = torch.Generator("cuda:0").manual_seed(seed)
    with torch.no_grad():
        norm.weight.add_(0.1 * torch.randn(K, generator=g, device="cuda:0"))
        head.weight.copy_(3 * K ** -0.5 * torch.randn(V, K, generator=g, device="cuda:0"))
    x = torch.randn(T, K, generator=g, device="cuda:0")
    add = None if add_dtype is None else torch.randn(T, K, generator=g, device="cuda:0").to(add_dtype)
    targets = torch.randint(0, V, (T,), generator=g, device="cuda:0")
    return norm, head, x, add, targets


@pytest.mark.parametrize("T,K,V", [(1, 64, 8), (17, 96, 200), (256, 128, 192), (255, 640, 1000), (257, 160, 392),   # edges of tiles, of quads of columns, two K steps
                                   (3000, 640, 32000),                                                              # several tiles a workgroup
                                   (700, 1536, 4104)])                                                              # the longest contraction
@pytest.mark.parametrize("add_dtype", [None, BF16, torch.float32])
def test_logits_with_their_loss(T, K, V, add_dtype):
    """The logits are bf16 of fp32 sums of products of the bf16 operands: off by 2^-8 of themselves, and by the sums' own rounding (K
    additions, below K 2^-24 of sum |h w|).  The loss is that of the stored logits: 2^-24 a term for exponentials, sums and logarithm, 1e-5."""
    from quartet_amd import kernels as Kn
    from quartet_amd.fused import logits_and_loss
    print(f"case logits {T}x{K}x{V}", flush=True)
    norm, head, x, add, targets = _head(T, K, V, add_dtype, T + K + V)
    targets[::5] = -1
    with torch.no_grad(), torch.autocast("cuda", dtype=BF16):
        assert Kn._lib.lib().qm_logits_loss_workspace_bytes(T, K, V)
        logits, loss = logits_and_loss(norm, head, x, add, targets)
        h = Kn.rmsnorm(x, norm.weight, norm.eps, add, BF16)
    assert logits.dtype == BF16 and logits.shape == (T, V) and loss.dtype == torch.float32
    h, w = h.double(), head.weight.detach().to(BF16).double()
    rows = torch.randperm(T, generator=torch.Generator().manual_seed(1))[:64].cuda()
    want = h[rows] @ w.T
    assert ((logits[rows].double() - want).abs() <= want.abs() * 2.0 ** -8 + K * 2.0 ** -24 * (h[rows].abs() @ w.abs().T)).all()
    if T > 1:
        ref = torch.nn.functional.cross_entropy(logits.double(), targets, ignore_index=-1)
        assert abs(float(loss) - float(ref)) < 1e-5 * max(1.0, abs(float(ref)))
    else:   # the only row is ignored: 0 / 0, as the library
        assert torch.isnan(loss)


@pytest.mark.parametrize("size", [20.0, 128.0, 1000.0, 1e5, 1e10, 1e38])
@pytest.mark.parametrize("T,V", [(64, 200), (256, 384)])   # edges, and whole tiles
def test_loss_of_large_logits(T, V, size):
    """Row by row, and whether the target is a row's largest class or not, the loss of the stored logits: differences to a row's largest logit round to
    2^-24 of themselves, as the terms and the sums do (1e-5 in all), however large the logits are.  Never negative beyond that."""
    from quartet_amd import kernels as Kn
    print(f"case large logits {T}x{V} {size}", flush=True)
    K, g = 64, torch.Generator("cuda:0").manual_seed(V)
    x, gain = torch.randn(T, K, generator=g, device="cuda:0"), torch.ones(K, device="cuda:0")
    weight = torch.randn(V, K, generator=g, device="cuda:0")
    weight[V // 2:] *= 0.999   # near ties, too
    weight[V // 2:] += 1e-3 * weight[: V - V // 2]
    top = (Kn.rmsnorm(x, gain, 1e-5, None, BF16).double() @ weight.to(BF16).double().T).abs().max()
    weight = (weight * (size / float(top))).contiguous()
    one = torch.full((T,), -1, dtype=torch.int64, device="cuda:0")
    logits, _ = Kn.logits_loss(x, gain, 1e-5, None, weight, one, -1)
    assert torch.isfinite(logits).all() and logits.double().abs().max() > 0.9 * size
    for row in (0, 1, 17, T - 1):
        for target in (int(logits[row].argmax()), int(logits[row].argmin()), 5):
            one.fill_(-1)
            one[row] = target
            again, loss = Kn.logits_loss(x, gain, 1e-5, None, weight, one, -1)
            want = float(torch.nn.functional.cross_entropy(logits[row:row + 1].double(), one[row:row + 1]))
            assert torch.equal(again, logits) and abs(float(loss) - want) <= 1e-5 * max(1.0, abs(want)), (row, target, float(loss), want)


@pytest.mark.parametrize("T,K,V,one_pass", [(1, 64, 8, True), (40, 768, 32768, True), (40, 768, 32776, False), (4607, 768, 32776, False), (4608, 768, 32776, True),
                                            (1536, 256, 262144, True), (1536, 256, 262152, False), (40, 800, 256, False), (300, 1536, 400, False)])
def test_which_logits_have_their_loss_in_the_same_pass(monkeypatch, T, K, V, one_pass):
    """Large weights, which the library rounds once per autocast region, and long contractions are the library's: its logits, bit for bit."""
    from quartet_amd import fused
    print(f"case route logits {T}x{K}x{V}", flush=True)
    calls, logits_loss = [], fused.kernels.logits_loss
    monkeypatch.setattr(fused.kernels, "logits_loss", lambda *a: calls.append(a) or logits_loss(*a))
    norm, head, x, add, targets = _head(T, K, V, BF16, V)
    with torch.no_grad(), torch.autocast("cuda", dtype=BF16):
        logits, loss = fused.logits_and_loss(norm, head, x, add, targets)
        assert len(calls) == one_pass and torch.isfinite(loss)
        if not one_pass:
            assert torch.equal(logits, head(fused.rmsnorm(norm, head, x, add)))


def test_logits_with_values_that_are_not_finite():
    """A row with an infinite and NaN logits, a target that is no class: the library's answer (NaN where it asserts)."""
    from quartet_amd.fused import logits_and_loss
    norm, head, x, _, targets = _head(300, 64, 400, None, 3)
    with torch.no_grad():
        norm.weight.fill_(1.0)
        head.weight.zero_()
        head.weight[:, 0] = 1.0
        x.zero_()
        x[:, 0] = 1.0
        head.weight[7, 1] = float("inf")
        x[5, 1] = -1.0   # class 7 of row 5: -inf; of the others 0 times inf, NaN
        with torch.autocast("cuda", dtype=BF16):
            logits, loss = logits_and_loss(norm, head, x, None, targets)
            assert torch.isnan(loss) and logits[5, 7] == -float("inf")
            kept = torch.full_like(targets, -1)
            kept[5] = 3
            _, loss = logits_and_loss(norm, head, x, None, kept)
            want = torch.nn.functional.cross_entropy(logits[5:6].double(), kept[5:6])
            assert abs(float(loss) - float(want)) < 1e-5
            head.weight[7, 1] = 0.0
            _, loss = logits_and_loss(norm, head, x, None, torch.full_like(targets, 400))
            assert torch.isnan(loss)


@pytest.mark.parametrize("T,V", [(64, 200), (256, 384)])   # edges, and whole tiles
def test_loss_of_rows_with_infinite_logits(T, V):
    """Rows of nothing but -inf, with a segment of -inf beside finite logits, with one +inf and one -inf, and a finite one, each by itself: the library's loss of the
    stored logits (NaN where it is NaN), within the 1e-5 of finite ones."""
    from quartet_amd import kernels as Kn
    print(f"case infinite logits {T}x{V}", flush=True)
    K, inf = 64, float("inf")
    x, gain, weight = torch.zeros(T, K, device="cuda:0"), torch.ones(K, device="cuda:0"), torch.zeros(V, K, device="cuda:0")
    g = torch.Generator("cuda:0").manual_seed(V)
    weight[:, :4] = torch.randn(V, 4, generator=g, device="cuda:0")
    x[:, 0] = 1.0
    big = 3e38   # finite in bf16; times the normalised x of 8 it overflows the fp32 sum
    weight[:, 4] = -big            # column 4: every class to -inf
    part = torch.arange(V, device="cuda:0") % 192 // 32
    first = (part == 0) | (part == 1) | (part == 4)   # the 96 columns of a tile that one wave has, whose sum is one part of the row's; the others
    weight[first, 5] = -big        # column 5: every first part of a row
    weight[~first, 6] = -big       # column 6: every second one
    weight[7, 7], weight[9, 8] = big, -big
    for row, column in ((1, 4), (2, 5), (3, 6), (4, 7), (5, 8)):
        x[row, 0], x[row, column] = 0.0, 1.0
    for row in (2, 3, 5):
        x[row, 1] = 1.0
    one = torch.full((T,), -1, dtype=torch.int64, device="cuda:0")
    logits, _ = Kn.logits_loss(x, gain, 1e-5, None, weight, one, -1)
    assert (logits[1] == -inf).all()
    for row, gone in ((2, first), (3, ~first)):
        assert (logits[row, gone] == -inf).all() and torch.isfinite(logits[row, ~gone]).all()
    assert logits[4, 7] == inf and logits[5, 9] == -inf and torch.isfinite(logits[6]).all() and not torch.isnan(logits).any()
    for row in range(1, 7):
        for target in (0, 7, 9, 100, V - 1):
            one.fill_(-1)
            one[row] = target
            _, loss = Kn.logits_loss(x, gain, 1e-5, None, weight, one, -1)
            want = torch.nn.functional.cross_entropy(logits[row:row + 1].double(), one[row:row + 1]).float()
            assert torch.allclose(loss, want, rtol=1e-5, atol=1e-5, equal_nan=True), (row, target, float(loss), float(want))


@pytest.mark.parametrize("T,K,V", [(300, 1536, 4104), (130, 4096, 1000)])
def test_longer_contractions_of_the_logits(T, K, V):
    """What the entry point takes beyond what the model is sent there with, to the bounds of ``test_logits_with_their_loss``."""
    from quartet_amd import kernels as Kn
    print(f"case logits {T}x{K}x{V}", flush=True)
    norm, head, x, add, targets = _head(T, K, V, BF16, K)
    with torch.no_grad():
        logits, loss = Kn.logits_loss(x, norm.weight, norm.eps, add, head.weight, targets, -1)
        h, w = Kn.rmsnorm(x, norm.weight, norm.eps, add, BF16).double(), head.weight.to(BF16).double()
    want = h @ w.T
    assert ((logits.double() - want).abs() <= want.abs() * 2.0 ** -8 + K * 2.0 ** -24 * (h.abs() @ w.abs().T)).all()
    ref = float(torch.nn.functional.cross_entropy(logits.double(), targets))
    assert abs(float(loss) - ref) < 1e-5 * max(1.0, abs(ref))


def test_logits_and_loss_take_the_modules_where_somebody_listens_or_asks_for_gradients():
    import torch.nn.functional as F
    from quartet_amd.fused import logits_and_loss, rmsnorm
    norm, head, x, add, targets = _head(70, 64, 96, BF16, 5)
    x, add, targets = x.view(2, 35, 64), add.view(2, 35, 64), targets.view(2, 35)
    with torch.autocast("cuda", dtype=BF16):
        apart = lambda: head(rmsnorm(norm, head, x, add))
        logits, loss = logits_and_loss(norm, head, x, add, targets)   # the head's weight asks for a gradient
        assert logits.requires_grad and loss.requires_grad
        with torch.no_grad():
            one, one_loss = logits_and_loss(norm, head, x, add, targets)
            assert one.shape == logits.shape and abs(float(one_loss) - float(F.cross_entropy(one.view(-1, 96).double(), targets.view(-1)))) < 1e-5
            seen = []
            handle = head.register_forward_hook(lambda *a: seen.append(1))
            got, _ = logits_and_loss(norm, head, x, add, targets)
            assert len(seen) == 1 and torch.equal(got, apart())
            handle.remove()
            biased = torch.nn.Linear(64, 96).to("cuda:0")
            assert torch.equal(logits_and_loss(norm, biased, x, add, targets)[0], biased(rmsnorm(norm, biased, x, add)))
            with pytest.raises(RuntimeError):
                logits_and_loss(norm, head, x, add, targets.t().contiguous().t())   # no view of these as one row
    with torch.no_grad():   # no autocast: fp32 logits
        assert logits_and_loss(norm, head, x, add, targets)[0].dtype == torch.float32


@pytest.mark.parametrize("B,S,heads,hs", [(1, 1, 5, 128), (3, 65, 2, 64), (2, 512, 5, 128), (1, 130, 12, 32)])
def test_attention_called_directly_is_the_chosen_one(B, S, heads, hs):
    import torch.nn.functional as F
    from quartet_amd.llama import _first_choice, _sdpa_choice
    g = torch.Generator("cuda:0").manual_seed(S)
    q, k, v = (torch.randn(B, S, heads, hs, generator=g, device="cuda:0").to(BF16).transpose(1, 2) for _ in range(3))
    with torch.no_grad():
        with _sdpa_choice("auto", q):
            want = F.scaled_dot_product_attention(q, k, v, attn_mask=None, dropout_p=0.0, is_causal=True)
        got = _first_choice("auto", q, k, v, 0.0)
        assert got is not None and got.shape == want.shape and got.stride() == want.stride() and torch.equal(got, want)
        assert _first_choice("default", q, k, v, 0.0) is None and _first_choice("auto", q, k, v, 0.1) is None
        assert _first_choice("auto", q.float(), k.float(), v.float(), 0.0) is None
        with torch.autocast("cuda", dtype=torch.float16):
            assert _first_choice("auto", q, k, v, 0.0) is None
    assert _first_choice("auto", q.requires_grad_(True), k, v, 0.0) is None
