// FP4 x FP4 "TN" product for at most 64 rows of A: the forward product of a layer that decodes one batch of sequences.
//
// What bounds it: W has to come in once (4096 x 4096: 8.9 MB, 1.8 us at this card's copy rate); everything else is latency.
// The tile kernels of gemm_tile.hip walk K through a ring in LDS with one barrier per 128 indices and put one workgroup on 32
// columns: 9.6 us at 8 x 4096 x 4096 and 19.6 us at 1 x 4096 x 11008, a chain of 32 (86) steps on half of the CUs.  Here a
// workgroup owns 16 columns (256 workgroups at N = 4096) and its waves share K among them, each with its own run of K steps
// whose operands go straight from memory into the registers of v_mfma_scale_f32_16x16x128_f8f6f4, four steps ahead and
// without a barrier: in the tiled layout one K step of 16 rows is 1 KiB in exactly that instruction's order (lane l: row
// l % 16, block l / 16 of 32 codes).  The waves' partial sums meet in LDS and are added in wave order, so results are
// reproducible; they differ from the tile kernels' in the order of the fp32 additions, which shows where a row's group scales
// span so many octaves that its sum is not exact in 24 bits (columns of 2^-8 .. 2^8: one bf16 result in 3 * 10^4).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gemm_common.h"
#include "quantize_group.h"

namespace qm {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kRowsDepth = 4;   // K steps requested ahead of the products

// The waves' partial sums in wave order.  Element e of a lane is column n0 + 4 * (lane / 16) + e of row lane % 16.
template <int TM, int WAVES, typename OutT>
__device__ __forceinline__ void add_waves(v4f (&partial)[WAVES][TM][64], const v4f (&acc)[TM], int wave, int lane, int n0, int M, int N, float alpha,
                                          OutT* __restrict__ c) {
    if (wave < WAVES) {
#pragma unroll
        for (int i = 0; i < TM; ++i) partial[wave][i][lane] = acc[i];
    }
    __syncthreads();
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
    add_waves<TM, WAVES>(partial, acc, wave, lane, n0, M, N, alpha, c);
}

// The same with the forward quantizer of x (Hadamard block 32, quest RTN) in front of the product, in every workgroup: the
// decoded batch is so small that quantizing it 256 times over costs no more time than doing it once in a launch of its own,
// and a layer call is one launch.  The codes lie in LDS as [K step][row][64 bytes], the scales as one byte per group; the
// weight's first eight K steps are on their way meanwhile.  Up to sixteen waves quantize, a group to a lane where that is enough
// for all; WAVES of them multiply.  With WAVES alone, 8 x 4096 x 4096 took its 1024 groups four to a lane, one after the other, each
// with its own wait for memory: 9.1 us, now 7.0.  Bit-identical to the two launches.
constexpr int kDecodeThreads = 1024;
template <int WAVES, typename T, typename OutT>
__global__ __launch_bounds__(kDecodeThreads) void linear_decode_kernel(const T* __restrict__ x, float rot_c, uint32_t sign_word,
                                                                    const uint8_t* __restrict__ b_codes, const uint8_t* __restrict__ b_scales, int M, int N,
                                                                    int I, int K, OutT* __restrict__ c) {
    __shared__ v4f partial[WAVES][1][64];
    extern __shared__ uint4 x_codes[];   // [K / 128][M][4], then M * K / 32 scale bytes in the same order
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int row = lane & 15, block = lane >> 4, shift = 8 * block;
    const int nk = K / kBK, groups = K / 32, real_groups = I / 32;
    const int n0 = (int)blockIdx.x * 16;
    const bool multiplies = wave < WAVES;
    const int first = multiplies ? wave * nk / WAVES : 0, end = multiplies ? (wave + 1) * nk / WAVES : 0;
    uint8_t* const x_scales = reinterpret_cast<uint8_t*>(x_codes + M * groups);

    const int b_row = n0 + row < N ? n0 + row : N - 1;
    const uint8_t* b_code = b_codes + (int64_t)n0 * (K / 2) + row * 64 + block * 16;
    const uint8_t* b_scale = b_scales + (int64_t)b_row * groups;
    struct Steps {
        uint4 b[kRowsDepth];
        uint32_t sb[kRowsDepth];
    };
    const auto request = [&](Steps& f, int s) {
#pragma unroll
        for (int d = 0; d < kRowsDepth; ++d) {
            const int k = s + d < end ? s + d : end - 1;
            f.b[d] = *reinterpret_cast<const uint4*>(b_code + (int64_t)k * 1024);
            f.sb[d] = *reinterpret_cast<const uint32_t*>(b_scale + k * 4);
        }
    };
    Steps f0, f1;
    if (first < end) {
        request(f0, first);
        request(f1, first + kRowsDepth);
    }
    for (int i = (int)threadIdx.x; i < M * groups; i += (int)blockDim.x) {
        const int r = i / groups, g = i - r * groups, at = ((g >> 2) * M + r) * 4 + (g & 3);
        GroupCodes o{};   // columns past the end: zero codes and scales
        if (g < real_groups) {
            float v[32];
            load_group<T>(x + (int64_t)r * I + g * 32, v);
            rotate_group(v, rot_c, sign_word);
            quantize_group_regs<QUEST_RTN, false>(v, 0, 0, o);
        }
        x_codes[at] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
        x_scales[at] = (uint8_t)o.scale_byte;
    }
    __syncthreads();
    v4f acc[1] = {v4f{0.0f, 0.0f, 0.0f, 0.0f}};
    const int a_row = row < M ? row : M - 1;
    const auto multiply = [&](const Steps& f, int s) {
#pragma unroll
        for (int d = 0; d < kRowsDepth; ++d) {
            if (s + d >= end) break;   // uniform
            const int at = ((s + d) * M + a_row) * 4 + block;
            const uint4 a = x_codes[at];
            const v8i bv = v8i{(int)f.b[d].x, (int)f.b[d].y, (int)f.b[d].z, (int)f.b[d].w, 0, 0, 0, 0};
            const v8i av = v8i{(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
            acc[0] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv, av, acc[0], 4, 4, 0, (int)(f.sb[d] >> shift), 0, (int)x_scales[at]);
        }
    };
    for (int s = first; s < end; s += 2 * kRowsDepth) {
        multiply(f0, s);
        if (s + 2 * kRowsDepth < end) request(f0, s + 2 * kRowsDepth);
        if (s + kRowsDepth < end) multiply(f1, s + kRowsDepth);
        if (s + 3 * kRowsDepth < end) request(f1, s + 3 * kRowsDepth);
    }
    add_waves<1, WAVES>(partial, acc, wave, lane, n0, M, N, 1.0f, c);
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

// One launch instead of two while a CU's share of quantizing is no more than 1024 groups, four per lane (about 5 us, what the
// quantizer's own launch takes): 8x4096x4096 7.0 us against 4.2 + 4.2 and 1x4096x11008 7.2 against 4.4 + 5.6, where a call's
// host time, which is what bounds both, falls from 12.5 to 10.3 us (and from 8.9 to 7.2 with fewer attribute look-ups)
bool linear_decode_serves(int64_t T, int64_t I, int64_t O) {
    if (!(T > 0 && T <= 16 && I > 0 && I % 32 == 0 && I < (1 << 20) && O >= 8 && O % 8 == 0 && O < (1 << 24))) return false;
    const int64_t per_cu = ((O + 15) / 16 + device_cus() - 1) / device_cus();
    return T * (padded_cols(I) / 32) * per_cu <= 1024;
}

hipError_t linear_decode(const void* x, int x_dtype, int64_t T, int64_t I, int64_t O, uint32_t sign_word, const uint8_t* w_codes,
                         const uint8_t* w_scales, void* y, int y_dtype, hipStream_t stream) {
    if (!linear_decode_serves(T, I, O)) return hipErrorInvalidValue;
    const int K = (int)padded_cols(I);
    const unsigned lds = (unsigned)(T * (K / 32) * 17);
    const float c = hadamard_scale(32, x_dtype);
    const dim3 grid((unsigned)((O + 15) / 16));
    const auto go = [&](auto waves, auto tx, auto ty) {   // as many waves as gemm_rows() takes: the same sums in the same order
        constexpr int W = decltype(waves)::value;
        const int64_t lanes = (T * (K / 32) + 63) / 64 * 64;
        const unsigned threads = (unsigned)(lanes < W * 64 ? W * 64 : lanes < kDecodeThreads ? lanes : kDecodeThreads);
        linear_decode_kernel<W, decltype(tx), decltype(ty)><<<grid, dim3(threads), lds, stream>>>(
            static_cast<const decltype(tx)*>(x), c, sign_word, w_codes, w_scales, (int)T, (int)O, (int)I, K, static_cast<decltype(ty)*>(y));
    };
    const auto typed = [&](auto waves) {
        if (x_dtype == BF16) { if (y_dtype == BF16) go(waves, uint16_t{}, uint16_t{}); else go(waves, uint16_t{}, float{}); }
        else { if (y_dtype == BF16) go(waves, float{}, uint16_t{}); else go(waves, float{}, float{}); }
    };
    if (K >= 64 * kBK) typed(std::integral_constant<int, 8>{});
    else typed(std::integral_constant<int, 4>{});
    return hipGetLastError();
}

}  // namespace qm
