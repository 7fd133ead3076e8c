"""Shared helpers for the parity tests: torch <-> oracle array conversion and synthetic inputs."""
import numpy as np
import torch


def to_oracle(t):
    """torch tensor (bf16/f32/u8, any device) -> numpy array in the oracle's convention (bf16 as uint16 bits)."""
    t = t.detach().cpu().contiguous()
    if t.dtype == torch.bfloat16:
        return t.view(torch.int16).numpy().view(np.uint16)
    return t.numpy()


def from_oracle_bf16(a):
    return torch.from_numpy(a.view(np.int16)).view(torch.bfloat16)


def sign_int(signs):
    """+-1 vector -> python int bit mask (bit j set = column j negated)."""
    m = 0
    for j, s in enumerate(signs.tolist()):
        if s < 0:
            m |= 1 << j
    return m


def make_input(rows, cols, dtype, seed, outlier_frac=1e-3, scale=1.0, zero_rows=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g) * scale
    if outlier_frac:
        m = torch.rand(rows, cols, generator=g) < outlier_frac
        sgn = torch.where(torch.rand(rows, cols, generator=g) < 0.5, -1.0, 1.0)
        x = torch.where(m, 1e3 * sgn * scale, x)
    if zero_rows:
        x[:zero_rows] = 0
    return x.to(dtype)


def product_is_cut(M, N, K):
    """Whether the library cuts the FP4 product into K ranges where it is offered scratch: over scales that spread, sums in another
    order than the whole product's round differently in fp32."""
    from quartet_amd import kernels
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    part = lambda rows, cols, lo, hi: torch.randint(lo, hi, (rows, cols), generator=g, dtype=torch.uint8, device="cuda")
    operands = (part(M, K // 2, 0, 256), part(M, K // 32, 112, 136), part(N, K // 2, 0, 256), part(N, K // 32, 112, 136))
    ranges, whole = (kernels.gemm_mxfp4_tn(*operands, 1.0, torch.float32, split_k=s) for s in (True, False))
    return not torch.equal(ranges, whole)
