"""Kernels that take tensors of 96 MiB and more past the caches: whole calls above that size against the same rows in calls below it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def parts(t, n=2):
    return [p.contiguous() for p in t.chunk(n)]


# the cooperative kernel's three widths (two, four and eight vectors a lane), a width that leaves lanes idle
@pytest.mark.parametrize("rows,cols", [(3074, 2048), (3001, 2112), (1537, 4096), (770, 8192)])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_rmsnorm_backward(rows, cols, dtype):
    """Rows do not depend on each other: the same bits.  The gain's gradient: fp32 sums of 1024 or fewer rows a partial sum, then of as many
    partial sums, in another order: 2^-24 of the absolute terms for each of at most 2048 additions, 40 of them at random signs."""
    print(f"case rmsnorm backward {rows}x{cols} {dtype}", flush=True)
    from quartet_amd import kernels as K
    assert rows * cols * 16 >= 96 << 20 > (rows + 1) // 2 * cols * 16
    gen = torch.Generator(device="cuda").manual_seed(rows)
    new = lambda *s, dt=F32: torch.randn(*s, generator=gen, device="cuda").to(dt)
    x, gy, skip, gain = new(rows, cols, dt=dtype), new(rows, cols, dt=BF16), new(rows, cols, dt=dtype), 1 + 0.1 * new(cols)
    factor = (x.float().square().mean(-1) + 1e-5).rsqrt()
    mask = torch.randint(0, 256, (rows, cols // 8), generator=gen, device="cuda", dtype=torch.uint8)
    run = lambda x, gy, skip, factor, mask: K.rmsnorm_backward(gy, x, gain, factor, mask, 0x5A5A1234, BF16, skip=skip, want_bf16_copy=True)
    whole, halves = run(x, gy, skip, factor, mask), [run(*p) for p in zip(*map(parts, (x, gy, skip, factor, mask)))]
    assert torch.equal(whole[0], torch.cat([h[0] for h in halves])) and torch.equal(whole[2], torch.cat([h[2] for h in halves]))
    unmasked = K.masked_hadamard_bwd(gy, 32, BF16, 0x5A5A1234, mask, F32)
    scale = (unmasked.double() * x.double() * factor.double()[:, None]).abs().sum(0)
    assert ((whole[1] - sum(h[1] for h in halves)).double().abs() <= 40 * 2.0 ** -24 * scale + 1e-30).all()


# of a bf16 x, by itself (6 bytes an element) and with a skip gradient and a copy (10)
@pytest.mark.parametrize("rows,cols,extra", [(8193, 2048, False), (4098, 4096, False), (4917, 2048, True), (1230, 8192, True)])
def test_rmsnorm_backward_of_bf16(rows, cols, extra):
    """Rows do not depend on each other: the same bits."""
    print(f"case rmsnorm backward of bf16 {rows}x{cols} {extra}", flush=True)
    from quartet_amd import kernels as K
    per = 10 if extra else 6
    assert rows * cols * per >= 96 << 20 > (rows + 1) // 2 * cols * per
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x, gy, skip = (torch.randn(rows, cols, generator=gen, device="cuda").to(BF16) for _ in range(3))
    gain = 1 + 0.1 * torch.randn(cols, generator=gen, device="cuda")
    factor = (x.float().square().mean(-1) + 1e-5).rsqrt()
    mask = torch.randint(0, 256, (rows, cols // 8), generator=gen, device="cuda", dtype=torch.uint8)
    run = lambda x, gy, skip, factor, mask: K.rmsnorm_backward(gy, x, gain, factor, mask, 0x5A5A1234, BF16, skip=skip if extra else None, want_bf16_copy=extra)
    whole, halves = run(x, gy, skip, factor, mask), [run(*p) for p in zip(*map(parts, (x, gy, skip, factor, mask)))]
    for i in (0, 2) if extra else (0,):
        assert torch.equal(whole[i], torch.cat([h[i] for h in halves]))


@pytest.mark.parametrize("rows,cols,hd,dtype", [(12289, 4096, 32, BF16), (6145, 4096, 64, F32), (24577, 2048, 128, BF16)])
def test_inverse_rotation(rows, cols, hd, dtype):
    print(f"case inverse rotation {rows}x{cols} hd={hd} {dtype}", flush=True)
    from quartet_amd import kernels as K
    g = torch.randn(rows, cols, generator=torch.Generator(device="cuda").manual_seed(hd), device="cuda").to(dtype)
    mask = torch.randint(0, 256, (rows, cols // 8), device="cuda", dtype=torch.uint8)
    assert g.numel() * g.element_size() >= 96 << 20
    run = lambda g, m: K.masked_hadamard_bwd(g, hd, BF16, 0x0F1E2D3C, m)
    assert torch.equal(run(g, mask), torch.cat([run(*p) for p in zip(parts(g), parts(mask))]))


# past 96 MiB (loads) and past 256 MiB (stores, too), a last wave that is not whole
@pytest.mark.parametrize("rows,cols,hd,dtype", [(12297, 4096, 32, BF16), (6145, 4160, 64, F32), (24577, 2048, 128, BF16), (32769, 4096, 64, BF16), (16385, 4224, 32, F32)])
@pytest.mark.parametrize("mode", ["QUEST_RTN", "ABSMAX_RTN"])
def test_quantizer_values(rows, cols, hd, dtype, mode):
    print(f"case quantizer values {rows}x{cols} hd={hd} {dtype} {mode}", flush=True)
    from quartet_amd import _lib, kernels as K
    x = torch.randn(rows, cols, generator=torch.Generator(device="cuda").manual_seed(hd), device="cuda").to(dtype)
    assert x.numel() * x.element_size() >= 96 << 20
    quest = mode == "QUEST_RTN"

    def run(x):
        values, mask = torch.empty_like(x), torch.zeros(x.shape[0], cols // 8, dtype=torch.uint8, device="cuda")
        rc = _lib.lib().qm_pseudo_quantize_mxfp4(x.data_ptr(), _lib.QM_BF16 if dtype == BF16 else _lib.QM_F32, *x.shape, hd, K.sign_words(0x0F1E2D3C), getattr(K, "QM_" + mode), 0,
                                                 mask.data_ptr() if quest else None, values.data_ptr(), None)
        _lib.check(rc, "qm_pseudo_quantize_mxfp4")
        return values, mask
    whole, halves = run(x), [run(p) for p in parts(x, 3)]
    for got, want in zip(whole, zip(*halves)):
        assert torch.equal(got, torch.cat(want))


@pytest.mark.parametrize("rows,classes,dtype", [(1573, 32000, BF16), (787, 32003, F32), (1600, 31999, BF16)])
def test_loss(rows, classes, dtype):
    """The mean of two halves' means: at most 16 + 10 + 2 fp32 additions of positive losses and a division, twice: 64 roundings."""
    print(f"case loss {rows}x{classes} {dtype}", flush=True)
    from quartet_amd import kernels as K
    gen = torch.Generator(device="cuda").manual_seed(classes)
    logits = torch.randn(rows, classes, generator=gen, device="cuda").to(dtype)
    targets = torch.randint(0, classes, (rows,), generator=gen, device="cuda")
    assert logits.numel() * logits.element_size() >= 96 << 20
    whole = float(K.cross_entropy(logits, targets, -1))
    halves = sum(float(K.cross_entropy(a, b, -1)) * len(b) for a, b in zip(parts(logits), parts(targets))) / rows
    assert abs(whole - halves) <= 64 * 2.0 ** -24 * abs(halves)


def test_loss_of_more_rows_than_a_grid_holds():
    """256 threads a row and fewer than 2^32 threads in a launch: the rows' losses past 2^23 and 2^24 are those of the rows by themselves."""
    from quartet_amd import _lib
    rows, classes = (1 << 24) + 3, 5
    print(f"case loss of {rows} rows", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(1)
    logits = torch.randn(rows, classes, generator=gen, device="cuda").to(BF16)
    targets = torch.randint(0, classes, (rows,), generator=gen, device="cuda")

    def run(at, n):
        losses, loss = torch.full((n,), -1.0, device="cuda"), torch.empty((), device="cuda")
        part, t = logits[at:at + n], targets[at:at + n]   # the same addresses
        rc = _lib.lib().qm_cross_entropy(part.data_ptr(), _lib.QM_BF16, t.data_ptr(), n, classes, -1, losses.data_ptr(), loss.data_ptr(), None)
        _lib.check(rc, "qm_cross_entropy")
        torch.cuda.synchronize()
        return losses, float(loss)
    losses, mean = run(0, rows)
    for at in (0, (1 << 23) - 4, 1 << 23, (1 << 24) - 4):
        assert torch.equal(losses[at:at + 7], run(at, 7)[0])
    assert bool((losses > 0).all())
    assert abs(mean - float(losses.double().mean())) <= ((rows >> 10) + 12) * 2.0 ** -24 * mean
