// FP4 x FP4 "TN" product for at most 64 rows of A: the forward product of a layer that decodes one batch of sequences.
//
// What bounds it: W has to come in once (4096 x 4096: 8.9 MB, 1.8 us at this card's copy rate); everything else is latency.
// The tile kernels of gemm_tile.hip walk K through a ring in LDS with one barrier per 128 indices and put one workgroup on 32
// columns: 9.6 us at 8 x 4096 x 4096 and 19.6 us at 1 x 4096 x 11008, a chain of 32 (86) steps on half of the CUs.  Here a
// workgroup owns 16 columns (256 workgroups at N = 4096) and its waves share K among them, each with its own run of K steps
// whose operands go straight from memory into the registers of v_mfma_scale_f32_16x16x128_f8f6f4, four steps ahead and
// without a barrier: in the tiled layout one K step of 16 rows is 1 KiB in exactly that instruction's order (lane l: row
// l % 16, block l / 16 of 32 codes).  The waves' partial sums meet in LDS and are added in wave order, so results are
// reproducible; they differ from the tile kernels' in the order of the fp32 additions.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_common.h"

namespace qm {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kRowsDepth = 4;   // K steps requested ahead of the products

// W's rows are the instruction's first operand: a lane ends up with four consecutive columns of c, of row l % 16
template <int TM, int WAVES, typename OutT>
__global__ __launch_bounds__(WAVES * 64) void gemm_mxfp4_tn_rows_kernel(const uint8_t* __restrict__ a_codes, const uint8_t* __restrict__ a_scales,
                                                                         const uint8_t* __restrict__ b_codes, const uint8_t* __restrict__ b_scales,
                                                                         int M, int N, int K, float alpha, OutT* __restrict__ c) {
    __shared__ v4f partial[WAVES][TM][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int row = lane & 15, block = lane >> 4, shift = 8 * block;
    const int nk = K / kBK, groups = K / 32;
    const int n0 = (int)blockIdx.x * 16;
    const int first = wave * nk / WAVES, end = (wave + 1) * nk / WAVES;   // this wave's K steps

    // rows past the end are read as the last one (a tiled operand's code rows exist up to the next multiple of 16)
    const int b_row = n0 + row < N ? n0 + row : N - 1;
    const uint8_t* b_code = b_codes + (int64_t)n0 * (K / 2) + row * 64 + block * 16;
    const uint8_t* b_scale = b_scales + (int64_t)b_row * groups;
    const uint8_t *a_code[TM], *a_scale[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int r = i * 16 + row < M ? i * 16 + row : M - 1;
        a_code[i] = a_codes + (int64_t)(r & ~15) * (K / 2) + (r & 15) * 64 + block * 16;
        a_scale[i] = a_scales + (int64_t)r * groups;
    }
    struct Steps {
        uint4 b[kRowsDepth], a[kRowsDepth][TM];
        uint32_t sb[kRowsDepth], sa[kRowsDepth][TM];
    };
    // steps s .. s + depth - 1 of this wave; past its end a repeat of the last one, which is not multiplied
    const auto request = [&](Steps& f, int s) {
#pragma unroll
        for (int d = 0; d < kRowsDepth; ++d) {
            const int k = s + d < end ? s + d : end - 1;
            f.b[d] = *reinterpret_cast<const uint4*>(b_code + (int64_t)k * 1024);
            f.sb[d] = *reinterpret_cast<const uint32_t*>(b_scale + k * 4);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                f.a[d][i] = *reinterpret_cast<const uint4*>(a_code[i] + (int64_t)k * 1024);
                f.sa[d][i] = *reinterpret_cast<const uint32_t*>(a_scale[i] + k * 4);
            }
        }
    };
    v4f acc[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const auto multiply = [&](const Steps& f, int s) {
#pragma unroll
        for (int d = 0; d < kRowsDepth; ++d) {
            if (s + d >= end) break;   // uniform
            const v8i bv = v8i{(int)f.b[d].x, (int)f.b[d].y, (int)f.b[d].z, (int)f.b[d].w, 0, 0, 0, 0};
            const int sb = (int)(f.sb[d] >> shift);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const v8i av = v8i{(int)f.a[d][i].x, (int)f.a[d][i].y, (int)f.a[d][i].z, (int)f.a[d][i].w, 0, 0, 0, 0};
                acc[i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv, av, acc[i], 4, 4, 0, sb, 0, (int)(f.sa[d][i] >> shift));
            }
        }
    };
    if (first < end) {   // fewer K steps than waves: some have none
        Steps f0, f1;
        request(f0, first);
        for (int s = first; s < end; s += 2 * kRowsDepth) {
            if (s + kRowsDepth < end) request(f1, s + kRowsDepth);
            multiply(f0, s);
            if (s + 2 * kRowsDepth < end) request(f0, s + 2 * kRowsDepth);
            if (s + kRowsDepth < end) multiply(f1, s + kRowsDepth);
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) partial[wave][i][lane] = acc[i];
    __syncthreads();
    // element e of a lane is column 4 * (lane / 16) + e of row lane % 16
    for (int t = (int)threadIdx.x; t < TM * 64; t += WAVES * 64) {
        const int i = t >> 6, l = t & 63, m = i * 16 + (l & 15), n = n0 + 4 * (l >> 4);
        v4f sum = partial[0][i][l];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) sum += partial[w][i][l];
        if (m >= M || n >= N) continue;   // N is a multiple of 8
        OutT* dst = c + (int64_t)m * N + n;
        const v4f v = v4f{sum[0] * alpha, sum[1] * alpha, sum[2] * alpha, sum[3] * alpha};
        if constexpr (sizeof(OutT) == 2) {
            const v2bf p0 = __builtin_convertvector(v2f{v[0], v[1]}, v2bf), p1 = __builtin_convertvector(v2f{v[2], v[3]}, v2bf);
            *reinterpret_cast<uint2*>(dst) = make_uint2(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1));
        } else {
            *reinterpret_cast<v4f*>(dst) = v;
        }
    }
}

template <int TM, int WAVES>
hipError_t launch_rows(const TileProduct& p, int c_dtype, hipStream_t stream) {
    const dim3 grid((unsigned)((p.N + 15) / 16)), block(WAVES * 64);
    if (c_dtype == BF16)
        gemm_mxfp4_tn_rows_kernel<TM, WAVES, uint16_t><<<grid, block, 0, stream>>>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, p.M, p.N, p.K,
                                                                                   p.alpha, static_cast<uint16_t*>(p.c));
    else
        gemm_mxfp4_tn_rows_kernel<TM, WAVES, float><<<grid, block, 0, stream>>>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, p.M, p.N, p.K, p.alpha,
                                                                                static_cast<float*>(p.c));
    return hipGetLastError();
}

}  // namespace

// Which products run here rather than on the tile kernels; us, tile kernel -> this one, weights cycled through memory.
// Up to 16 rows always: 1x4096x11008 20.1 -> 8.2, 8x4096x4096 9.6 -> 4.9, 16x512x8192 15.2 -> 7.2, 16x640x640 4.3 -> 4.2,
// 16x11008x4096 11.0 -> 10.6, 16x11008x11008 23.8 -> 21.1.
// More rows while every CU has at most one workgroup (each reads all of A): 17x4096x4096 9.6 -> 5.6, 64x4096x4096 10.4 -> 9.4,
// 64x2048x11008 22.3 -> 18.6, but 32x6144x4096 9.8 -> 10.5, 64x6144x4096 10.6 -> 17.4.  Up to 32 rows also where K is short
// enough for that not to matter: 32x8192x1536 6.0 -> 4.9, but 64x8192x1536 6.2 -> 7.5.
bool gemm_rows_serves(const TileProduct& p) {
    const bool kind = p.M > 0 && p.M <= 64 && p.N >= 8 && p.N % 8 == 0 && p.K > 0 && p.K % kBK == 0 && p.a_tiled && p.b_tiled && !p.mask &&
                      !p.b_e5m2 && (reinterpret_cast<uintptr_t>(p.c) & 15) == 0;
    return kind && (p.M <= 16 || p.N <= 16 * device_cus() || (p.M <= 32 && p.K <= 2048));
}

// Waves: four, one per SIMD (8x8192x1536: 4.3 against 5.2 with eight, 64x4096x4096 9.4 / 10.8); eight where a long K leaves each
// of them enough steps and few rows enough registers (1x4096x11008 8.2 against 8.7, 16x11008x11008 21.1 / 22.3)
hipError_t gemm_rows(const TileProduct& p, int c_dtype, hipStream_t stream) {
    if (!gemm_rows_serves(p)) return hipErrorInvalidValue;
    if (p.M <= 16) return p.K >= 64 * kBK ? launch_rows<1, 8>(p, c_dtype, stream) : launch_rows<1, 4>(p, c_dtype, stream);
    if (p.M <= 32) return launch_rows<2, 4>(p, c_dtype, stream);
    return launch_rows<4, 4>(p, c_dtype, stream);
}

}  // namespace qm
