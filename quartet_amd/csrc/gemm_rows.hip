// FP4 x FP4 "TN" product for at most 64 rows of A: the forward product of a layer that decodes one batch of sequences.
//
// What bounds it: W has to come in once (4096 x 4096: 8.9 MB, 1.8 us at this card's copy rate); everything else is latency.
// The tile kernels of gemm_tile.hip walk K through a ring in LDS with one barrier per 128 indices and put one workgroup on 32
// columns: 9.6 us at 8 x 4096 x 4096 and 19.6 us at 1 x 4096 x 11008, a chain of 32 (86) steps on half of the CUs.  Here a
// workgroup owns 16 columns (256 workgroups at N = 4096; more rows or columns: rows_tile()) and its waves share K among them, each with its own run of K steps
// whose operands go straight from memory into the registers of v_mfma_scale_f32_16x16x128_f8f6f4, four to eight steps ahead and
// without a barrier: in the tiled layout one K step of 16 rows is 1 KiB in exactly that instruction's order (lane l: row
// l % 16, block l / 16 of 32 codes).  The waves' partial sums meet in LDS and are added in wave order, so results are
// reproducible; they differ from the tile kernels' in the order of the fp32 additions, which shows where a row's group scales
// span so many octaves that its sum is not exact in 24 bits (columns of 2^-8 .. 2^8: one bf16 result in 3 * 10^4).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gemm_common.h"
#include "quantize_group.h"
#include "scale_requests.h"

namespace qm {

// With scales requested a step at a time, which touch as many cache lines as the codes do, and each request behind a condition (waits below), it
// took, us MxNxK: 16x4096x4096 5.2 (now 3.9), 16x11008x4096 10.3 (6.4), 32x4096x4096 6.5 (4.4), 64x4096x4096 9.3 (5.3), 64x4096x11008 14.6 (8.9), 64x1536x8192
// 15.7 (6.5); with the quantizer in it 1x11008x4096 8.2 (7.3, in wider workgroups 6.7), 8x4096x4096 6.3 (6.1).
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kRowsDepth = 4;   // K steps requested at a time
struct Scales {   // of a row's groups in that many steps: 4-byte aligned, as rows of a multiple of 128 have them
    uint32_t w[kRowsDepth];
};
__device__ __forceinline__ Scales moved(const Scales& v, int by) {   // `by` steps on
    const uint32_t w0 = v.w[0], w1 = v.w[1], w2 = v.w[2], w3 = v.w[3];
    return Scales{{by == 0 ? w0 : by == 1 ? w1 : by == 2 ? w2 : w3, by == 0 ? w1 : by == 1 ? w2 : w3, by == 0 ? w2 : w3, w3}};
}

// The waves' partial sums in wave order.  Element e of a lane of tile (i, j) is column n0 + 16 j + 4 * (lane / 16) + e of row m0 + 16 i + lane % 16.
template <int TM, int TN, int WAVES, typename OutT>
__device__ __forceinline__ void add_waves(const v4f (&partial)[WAVES][TM * TN][64], int threads, int m0, int n0, int M, int N, float alpha, OutT* __restrict__ c) {
    __syncthreads();
    for (int t = (int)threadIdx.x; t < TM * TN * 64; t += threads) {
        const int tile = t >> 6, l = t & 63, m = m0 + tile / TN * 16 + (l & 15), n = n0 + tile % TN * 16 + 4 * (l >> 4);
        v4f sum = partial[0][tile][l];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) sum += partial[w][tile][l];
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
template <int TM, int TN, int WAVES, typename OutT>
__global__ __launch_bounds__(WAVES * 64) void gemm_mxfp4_tn_rows_kernel(const uint8_t* __restrict__ a_codes, const uint8_t* __restrict__ a_scales,
                                                                         const uint8_t* __restrict__ b_codes, const uint8_t* __restrict__ b_scales,
                                                                         int M, int N, int K, float alpha, OutT* __restrict__ c) {
    __shared__ v4f partial[WAVES][TM * TN][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int row = lane & 15, block = lane >> 4, shift = 8 * block;
    const int nk = K / kBK, groups = K / 32;
    const int n0 = (int)blockIdx.x * 16 * TN, m0 = (int)blockIdx.y * 16 * TM;
    const int first = wave * nk / WAVES, end = (wave + 1) * nk / WAVES;   // this wave's K steps

    // A tiled operand's code rows exist up to the next multiple of 16: blocks of 16 rows past that are read as the last one, and of scales
    // rows past the end as the last row.
    const uint32_t in_block = (uint32_t)(row * 64 + block * 16);
    const uint8_t *a_code[TM], *a_scale[TM], *b_code[TN], *b_scale[TN];   // uniform
    uint32_t a_row[TM], b_row[TN];                                       // the lane's row of scales behind them
    const auto block_of = [&](int from, int rows, const uint8_t* codes, const uint8_t* scales, const uint8_t*& code, const uint8_t*& scale, uint32_t& at) {
        from = from < rows ? from : (rows - 1) & ~15;
        code = codes + (int64_t)from * (K / 2);
        scale = scales + (int64_t)from * groups;
        at = (uint32_t)(from + row < rows ? row : rows - 1 - from) * (uint32_t)groups;
    };
#pragma unroll
    for (int i = 0; i < TM; ++i) block_of(m0 + i * 16, M, a_codes, a_scales, a_code[i], a_scale[i], a_row[i]);
#pragma unroll
    for (int j = 0; j < TN; ++j) block_of(n0 + j * 16, N, b_codes, b_scales, b_code[j], b_scale[j], b_row[j]);
    struct Steps {
        Scales sa[TM], sb[TN];
        uint4 a[kRowsDepth][TM], b[kRowsDepth][TN];
    };
    // Steps s .. s + depth - 1 of this wave; past its end sixteen bytes of the last one for all lanes, which cost one request and are not multiplied.
    // Their scales in one request, which at a row's end begins up to three steps earlier (multiply_last): in rows of fewer steps in front of the
    // row, which in a packed operand's first row is among its codes (scale_requests.h; what is not packed so does not come here).
    const auto request = [&](Steps& f, int s) {
        const int from = 4 * (s + kRowsDepth <= nk ? s : nk - kRowsDepth);
#pragma unroll
        for (int j = 0; j < TN; ++j) f.sb[j] = *reinterpret_cast<const Scales*>(b_scale[j] + from + b_row[j]);
#pragma unroll
        for (int i = 0; i < TM; ++i) f.sa[i] = *reinterpret_cast<const Scales*>(a_scale[i] + from + a_row[i]);
#pragma unroll
        for (int d = 0; d < kRowsDepth; ++d) {
            const int64_t at = (int64_t)(s + d < end ? s + d : end - 1) * 1024;
            const uint32_t off = s + d < end ? in_block : 0u;
#pragma unroll
            for (int j = 0; j < TN; ++j) f.b[d][j] = *reinterpret_cast<const uint4*>(b_code[j] + at + off);
#pragma unroll
            for (int i = 0; i < TM; ++i) f.a[d][i] = *reinterpret_cast<const uint4*>(a_code[i] + at + off);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    v4f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const auto multiply = [&](const Steps& f, int steps) {
#pragma unroll
        for (int d = 0; d < kRowsDepth; ++d) {
            if (d >= steps) break;   // uniform
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const v8i av = v8i{(int)f.a[d][i].x, (int)f.a[d][i].y, (int)f.a[d][i].z, (int)f.a[d][i].w, 0, 0, 0, 0};
                const int sa = (int)(f.sa[i].w[d] >> shift);
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const v8i bv = v8i{(int)f.b[d][j].x, (int)f.b[d][j].y, (int)f.b[d][j].z, (int)f.b[d][j].w, 0, 0, 0, 0};
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv, av, acc[i][j], 4, 4, 0, (int)(f.sb[j].w[d] >> shift), 0, sa);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto multiply_last = [&](Steps& f, int s) {
        const int by = s + kRowsDepth <= nk ? 0 : s + kRowsDepth - nk;
#pragma unroll
        for (int j = 0; j < TN; ++j) f.sb[j] = moved(f.sb[j], by);
#pragma unroll
        for (int i = 0; i < TM; ++i) f.sa[i] = moved(f.sa[i], by);
        multiply(f, end - s);
    };
    // Requests without a condition of their own: behind one that may or may not have been made, the compiler waits for what is older as if it had not
    // been, which is for everything.
    if (first < end) {   // fewer K steps than waves: some have none
        Steps f0, f1;
        if (end - first <= kRowsDepth) {
            request(f0, first);
            multiply_last(f0, first);
        } else {
            request(f0, first);
            request(f1, first + kRowsDepth);
            int s = first;
#pragma unroll 1
            for (; s + 2 * kRowsDepth < end; s += 2 * kRowsDepth) {
                multiply(f0, kRowsDepth);
                request(f0, s + 2 * kRowsDepth);
                multiply(f1, kRowsDepth);
                request(f1, s + 3 * kRowsDepth);
            }
            multiply_last(f0, s);
            multiply_last(f1, s + kRowsDepth);
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) partial[wave][i * TN + j][lane] = acc[i][j];
    add_waves<TM, TN, WAVES>(partial, WAVES * 64, m0, n0, M, N, alpha, c);
}

// The same with the forward quantizer of x (Hadamard block 32, quest RTN) in front of the product, in every workgroup: the
// decoded batch is so small that quantizing it 256 times over costs no more time than doing it once in a launch of its own,
// and a layer call is one launch.  The codes lie in LDS as [K step][row][64 bytes], the scales as one byte per group; the
// weight's first eight K steps are on their way meanwhile.  Up to sixteen waves quantize, a group to a lane where that is enough
// for all; WAVES x TN of them multiply.  With WAVES alone, 8 x 4096 x 4096 took its 1024 groups four to a lane, one after the other, each
// with its own wait for memory: 9.1 us, now 6.1 behind another one and 6.7 to 7 by itself.  Bit-identical to the two launches.
// TN: 16 columns each, with waves of their own, so that what a wave holds and adds is the same for any TN.  Wide layers have as many as leave one
// workgroup to a CU (decode_columns()): with 16 columns a workgroup their CUs quantize all of x two to four times over.
constexpr int kDecodeThreads = 1024;
template <int WAVES, int TN, typename T, typename OutT>
__global__ __launch_bounds__(kDecodeThreads) void linear_decode_kernel(const T* __restrict__ x, float rot_c, uint32_t sign_word,
                                                                    const uint8_t* __restrict__ b_codes, const uint8_t* __restrict__ b_scales, int M, int N,
                                                                    int I, int K, OutT* __restrict__ c) {
    __shared__ v4f partial[WAVES][TN][64];
    extern __shared__ uint4 x_codes[];   // [K / 128][M][4], then M * K / 32 scale bytes in the same order
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int row = lane & 15, block = lane >> 4, shift = 8 * block;
    const int nk = K / kBK, groups = K / 32, real_groups = I / 32;
    const int n0 = (int)blockIdx.x * 16 * TN;
    const bool multiplies = wave < WAVES * TN;
    const int share = wave % WAVES, column = wave / WAVES;   // of K, and which 16 columns
    const int first = multiplies ? share * nk / WAVES : 0, end = multiplies ? (share + 1) * nk / WAVES : 0;
    uint8_t* const x_scales = reinterpret_cast<uint8_t*>(x_codes + M * groups);

    const uint32_t in_block = (uint32_t)(row * 64 + block * 16);
    int from = n0 + 16 * column;   // past the end the last 16 rows of W, which are not stored
    from = from < N ? from : (N - 1) & ~15;
    const uint8_t* b_code = b_codes + (int64_t)from * (K / 2);
    b_scales += (int64_t)from * groups;
    const uint32_t b_scale = (uint32_t)(from + row < N ? row : N - 1 - from) * (uint32_t)groups;
    struct Steps {
        Scales sb;
        uint4 b[kRowsDepth];
    };
    const auto request = [&](Steps& f, int s) {   // as above
        f.sb = *reinterpret_cast<const Scales*>(b_scales + 4 * (s + kRowsDepth <= nk ? s : nk - kRowsDepth) + b_scale);
#pragma unroll
        for (int d = 0; d < kRowsDepth; ++d)
            f.b[d] = *reinterpret_cast<const uint4*>(b_code + (int64_t)(s + d < end ? s + d : end - 1) * 1024 + (s + d < end ? in_block : 0u));
        __builtin_amdgcn_sched_barrier(0);
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
    v4f acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const int a_row = row < M ? row : M - 1;
    const auto multiply = [&](const Steps& f, int s, int steps) {
#pragma unroll
        for (int d = 0; d < kRowsDepth; ++d) {
            if (d >= steps) break;   // uniform
            const int at = ((s + d) * M + a_row) * 4 + block;
            const uint4 a = x_codes[at];
            const v8i bv = v8i{(int)f.b[d].x, (int)f.b[d].y, (int)f.b[d].z, (int)f.b[d].w, 0, 0, 0, 0};
            const v8i av = v8i{(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
            acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv, av, acc, 4, 4, 0, (int)(f.sb.w[d] >> shift), 0, (int)x_scales[at]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto multiply_last = [&](Steps& f, int s) {
        f.sb = moved(f.sb, s + kRowsDepth <= nk ? 0 : s + kRowsDepth - nk);
        multiply(f, s, end - s);
    };
    int s = first;
#pragma unroll 1
    for (; s + 2 * kRowsDepth < end; s += 2 * kRowsDepth) {
        multiply(f0, s, kRowsDepth);
        request(f0, s + 2 * kRowsDepth);
        multiply(f1, s + kRowsDepth, kRowsDepth);
        request(f1, s + 3 * kRowsDepth);
    }
    multiply_last(f0, s);
    multiply_last(f1, s + kRowsDepth);
    if (multiplies) partial[share][column][lane] = acc;
    add_waves<1, TN, WAVES>(partial, (int)blockDim.x, 0, n0, M, N, 1.0f, c);
}
template <int TM, int TN, int WAVES>
hipError_t launch_rows(const TileProduct& p, int c_dtype, hipStream_t stream) {
    const dim3 grid((unsigned)((p.N + 16 * TN - 1) / (16 * TN)), (unsigned)((p.M + 16 * TM - 1) / (16 * TM))), block(WAVES * 64);
    if (c_dtype == BF16)
        gemm_mxfp4_tn_rows_kernel<TM, TN, WAVES, uint16_t><<<grid, block, 0, stream>>>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, p.M, p.N, p.K,
                                                                                   p.alpha, static_cast<uint16_t*>(p.c));
    else
        gemm_mxfp4_tn_rows_kernel<TM, TN, WAVES, float><<<grid, block, 0, stream>>>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, p.M, p.N, p.K, p.alpha,
                                                                                static_cast<float*>(p.c));
    return hipGetLastError();
}

}  // namespace

// Tiles of 16 TM rows and 16 TN columns for four waves.  A workgroup requests (TM + TN) KiB a K step and little else bounds it, so the best tile is
// the one whose workgroups bring in least per CU, in whole rounds of one to a CU: 24 ns a KiB, and beyond that what larger tiles take to start and
// end.  us, by tile (1 x 1, 2 x 1, 2 x 2, 2 x 4; MxNxK): 32x2048x2048 2.7, 3.0, 3.3, 4.5; 32x4096x4096 5.2, 4.5, 5.2, 7.1; 64x4096x4096 -, 6.5, 5.3, 7.1;
// 64x4096x11008 -, 12.7, 9.3, 13.2; 64x8192x4096 -, 10.5, 8.5, 7.3; 32x11008x4096 10.6, 8.5, 8.6, 7.6.  16x11008x4096 with 1 x 1 6.7, with 1 x 4 6.1.
enum RowsTile : int { ROWS_1x1, ROWS_2x1, ROWS_2x2, ROWS_1x4, ROWS_2x4 };
RowsTile rows_tile(const TileProduct& p) {
    constexpr struct { int tm, tn; double start; } kTiles[] = {{1, 1, 0.0}, {2, 1, 0.15}, {2, 2, 0.25}, {1, 4, 0.25}, {2, 4, 0.55}};
    const int64_t cus = device_cus();
    int best = 0;
    double least = 1e30;
    for (int t = 0; t < 5; ++t) {
        const int64_t workgroups = (int64_t)((p.M + 16 * kTiles[t].tm - 1) / (16 * kTiles[t].tm)) * ((p.N + 16 * kTiles[t].tn - 1) / (16 * kTiles[t].tn));
        const double us = kTiles[t].start + 0.024 * (double)((workgroups + cus - 1) / cus * (kTiles[t].tm + kTiles[t].tn)) * (p.K / kBK);
        if (us < least) {
            least = us;
            best = t;
        }
    }
    return (RowsTile)best;
}

// Which products (MxNxK) run here rather than on the tile kernels: up to 16 rows all; up to 32 while their 2 x 4 tiles are at most three on four CUs, or
// K is short; up to 64 while those are at most one on a CU.  us, tile kernel -> this one: 1x4096x11008 20.1 -> 5.9, 16x11008x4096 11.0 -> 6.4,
// 17x4096x4096 9.6 -> 4.3, 32x8192x4096 7.8 -> 5.7, 32x11008x11008 15.9 -> 15.1, 64x8192x1536 4.9 -> 4.5, 64x8192x4096 7.9 -> 7.2; but 32x16384x4096
// 8.7 -> 9.1, 64x11008x4096 8.3 -> 9.4.
bool gemm_rows_serves(const TileProduct& p) {
    const bool kind = p.M > 0 && p.M <= 64 && p.N >= 8 && p.N % 8 == 0 && p.K > 0 && p.K % kBK == 0 && p.a_tiled && p.b_tiled && !p.mask &&
                      !p.b_e5m2 && (reinterpret_cast<uintptr_t>(p.c) & 15) == 0 && scale_requests_in_operand(p.a_codes, p.a_scales, p.M, p.K) &&
                      scale_requests_in_operand(p.b_codes, p.b_scales, p.N, p.K);
    const int64_t tiles = ((int64_t)p.N + 63) / 64;
    return kind && (p.M <= 16 || (p.M <= 32 ? p.K <= 2048 || 4 * tiles <= 3 * device_cus() : 2 * tiles <= device_cus()));
}

// Waves: four, one per SIMD (8x8192x1536 3.5, with eight 3.6; 64x4096x4096 5.3 and 5.6); eight where few rows meet a long K, whose sums are then of
// shorter chains (16x4096x11008 6.4 and, with four, 6.0)
hipError_t gemm_rows(const TileProduct& p, int c_dtype, hipStream_t stream) {
    if (!gemm_rows_serves(p)) return hipErrorInvalidValue;
    if (p.M <= 16 && p.K >= 64 * kBK) return launch_rows<1, 1, 8>(p, c_dtype, stream);
    switch (rows_tile(p)) {
        case ROWS_1x1: return launch_rows<1, 1, 4>(p, c_dtype, stream);
        case ROWS_2x1: return launch_rows<2, 1, 4>(p, c_dtype, stream);
        case ROWS_2x2: return launch_rows<2, 2, 4>(p, c_dtype, stream);
        case ROWS_1x4: return launch_rows<1, 4, 4>(p, c_dtype, stream);
        default: return launch_rows<2, 4, 4>(p, c_dtype, stream);
    }
}

// Columns of a workgroup, in sixteens: as many as it takes for one workgroup to a CU, of which sixteen waves are the most.  us by columns / 16 (1, 2, 3, 4;
// MxNxK): 8x4096x4096 6.7, 6.4, 6.8, 7.3; 8x8192x2048 6.6, 5.1, 5.3, 5.4; 12x4608x2048 8.4, 5.3, 6.0, 6.2; 8x11008x4096 15.8, 12.2, 8.1, 8.5; 16x11008x1152 11.5,
// 8.5, 5.8, 5.9; 1x16384x2048 6.3, 6.0, 7.9, 5.7; 4x8192x8192 (eight waves to K) 13.1, 9.7.  Of few groups equal: 1x11008x640 4.2, 4.5, 4.3, 4.5.
int decode_columns(int64_t O, int64_t K) {
    const int64_t blocks = (O + 15) / 16, most = K >= 64 * kBK ? 2 : 4, need = (blocks + device_cus() - 1) / device_cus();
    return (int)(need < most ? need : most);
}

// One launch instead of two while a CU's share of quantizing is no more than 1024 groups, one to a lane (about 3 us; the quantizer's own
// launch takes 4): us in two launches and in one, 8x4096x4096 6.7 and 6.1 to 6.7, 8x11008x4096 9.8 and 8.1, 4x11008x4096 9.5 and 6.9, 16x11008x2048 8.1 and
// 6.6, 1x4096x4096 6.7 and 4.7, 2x11008x11008 (1376 groups) 17.9 and 17.4; a call's host time, which bounds most of these, falls from 10.6 to 7.2
bool linear_decode_serves(int64_t T, int64_t I, int64_t O) {
    if (!(T > 0 && T <= 16 && I > 0 && I % 32 == 0 && I < (1 << 20) && O >= 8 && O % 8 == 0 && O < (1 << 24))) return false;
    const int64_t K = padded_cols(I), columns = 16 * decode_columns(O, K);
    const int64_t per_cu = ((O + columns - 1) / columns + device_cus() - 1) / device_cus();
    return T * (K / 32) * per_cu <= 1024;
}

hipError_t linear_decode(const void* x, int x_dtype, int64_t T, int64_t I, int64_t O, uint32_t sign_word, const uint8_t* w_codes,
                         const uint8_t* w_scales, void* y, int y_dtype, hipStream_t stream) {
    if (!linear_decode_serves(T, I, O) || !scale_requests_in_operand(w_codes, w_scales, O, padded_cols(I))) return hipErrorInvalidValue;
    const int K = (int)padded_cols(I), columns = decode_columns(O, K);
    const unsigned lds = (unsigned)(T * (K / 32) * 17);
    const float c = hadamard_scale(32, x_dtype);
    const dim3 grid((unsigned)((O + 16 * columns - 1) / (16 * columns)));
    const auto go = [&](auto waves, auto tn, auto tx, auto ty) {   // as many waves to K as gemm_rows() takes: the same sums in the same order
        constexpr int W = decltype(waves)::value, TN = decltype(tn)::value;
        const int64_t lanes = (T * (K / 32) + 63) / 64 * 64;
        const unsigned threads = (unsigned)(lanes < W * TN * 64 ? W * TN * 64 : lanes < kDecodeThreads ? lanes : kDecodeThreads);
        linear_decode_kernel<W, TN, decltype(tx), decltype(ty)><<<grid, dim3(threads), lds, stream>>>(
            static_cast<const decltype(tx)*>(x), c, sign_word, w_codes, w_scales, (int)T, (int)O, (int)I, K, static_cast<decltype(ty)*>(y));
    };
    const auto typed = [&](auto waves, auto tn) {
        if (x_dtype == BF16) { if (y_dtype == BF16) go(waves, tn, uint16_t{}, uint16_t{}); else go(waves, tn, uint16_t{}, float{}); }
        else { if (y_dtype == BF16) go(waves, tn, float{}, uint16_t{}); else go(waves, tn, float{}, float{}); }
    };
    if (K >= 64 * kBK) {
        const std::integral_constant<int, 8> waves;
        if (columns == 1) typed(waves, std::integral_constant<int, 1>{});
        else typed(waves, std::integral_constant<int, 2>{});
    } else {
        const std::integral_constant<int, 4> waves;
        if (columns == 1) typed(waves, std::integral_constant<int, 1>{});
        else if (columns == 2) typed(waves, std::integral_constant<int, 2>{});
        else if (columns == 3) typed(waves, std::integral_constant<int, 3>{});
        else typed(waves, std::integral_constant<int, 4>{});
    }
    return hipGetLastError();
}

}  // namespace qm
