// FP4 x FP4 and bf16 x bf16 "TN" products on tiles of 256 x 192, two workgroups to a CU: a plain bf16 result of two tiled operands.
//
// The persistent kernel of gemm.hip owns a CU with one workgroup and a tile of 256 x 256, and the smaller shapes of gemm_tile.hip read 1.5 times
// its bytes from LDS per product.  In between, a wave of 128 x 96 holds 192 accumulators, which leaves 64 of the 256 registers that two waves
// on a SIMD have, and reads 1.17 times its bytes.  Tiles three quarters as large fill a chip's last round better, and a workgroup's barriers,
// first fill and epilogue are covered by the other one of its CU.
//
// What bounds it: the request of a K step is on its way for one step only (two slots of 28 KiB; three do not fit twice into 160 KiB), and at
// long contractions the power limit.  On zero codes, where that limit is out of reach, a CU takes 2150 cycles for a K step of both of its tiles (1536 by
// the matrix instructions, 1344 of LDS accesses).  us behind a copy, the faster of the other kernels and this one: 16384 x 1536 x 4096 57.2 and
// 52.5, 8192 x 4608 x 1536 40 and 36.6, 16832 x 9280 x 2176 204 and 180; traced inside a step 67.3 -> 59.9, 47.5 -> 39 and (16384 x 4608 x 1536) 78.0 ->
// 75.7; the steps 409.6 -> 409.4, 189.5 -> 185.8 and 438.5 -> 429.8, since part of what a product gains the power limit takes elsewhere.
// Tried: fragments read a half step ahead across the barrier (scratch memory; 5 % slower), requests ahead of the products instead of among
// them (4 % slower).
//
// The same with bf16 operands makes the logits of an evaluated model, whose workgroups also take the exponentials for their loss while the other one
// of the CU multiplies: no pass of its own over logits that are larger than the caches.  Bound by the matrix instructions at the power limit and the last,
// partial round of tiles: 4096 x 32000 x 640 166 us (153 without the exponentials; the library's product 158 and the loss's pass 49), and from 1536
// on by its two slots (4096 x 32000 x 1536 339; the library's product 300), which the model leaves to the library, as it does weights that cost more to round
// than that pass (fused.py).  An evaluated 30 M model of 8 x 512 tokens 884 -> 847 us when it came; exponentials of differences, for the loss of large
// logits, take 3 us of that back.
// Row-major operands, 64 bytes of a row at a time, took 176 and 380.
//
// The order of additions over K is that of gemm.hip and gemm_tile.hip: the same bits.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gemm_common.h"

namespace qm {

namespace {

constexpr int kTwoM = 256, kTwoN = 192, kTwoTM = 4, kTwoTN = 3;   // four waves, two by two; 32 x 32 blocks of a wave
constexpr int kTwoBOff = kTwoM * kRowBytes, kTwoSlot = (kTwoM + kTwoN) * kRowBytes;
constexpr int kTwoScales = 2 * kTwoSlot, kTwoScaleBuf = (kTwoM + kTwoN) * 16;   // 16 bytes a row: the scales of four K steps, two such blocks
constexpr int kTwoLds = kTwoScales + 2 * kTwoScaleBuf;
static_assert(2 * kTwoLds <= 160 * 1024, "two workgroups to a CU");

// requests at M0 + offset, which moves source and destination alike: the source of request I is given I KiB short
__device__ __forceinline__ void two_lds_base(uint32_t lds) { asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" ::"s"(lds)); }
template <int I>
__device__ __forceinline__ void two_request(const uint8_t* base, uint32_t lane_off) {
    asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" ::"v"(lane_off), "s"(base), "i"(I * 1024) : "memory");
}
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
constexpr float kLog2e = 1.44269504088896340736f;
__device__ __forceinline__ v8i two_operand(const uint4& q) { return v8i{(int)q.x, (int)q.y, (int)q.z, (int)q.w, 0, 0, 0, 0}; }

// EDGES: M or N is no multiple of the tile's.  Rows past the end repeat others, and nothing of theirs is stored.
// BF16: both operands are bf16 in blocks of 16 rows and 32 elements, [R / 16][K / 32][16][64 bytes]: 32 elements in the place of 128 FP4 codes, no scales,
// no alpha.  Beside the result it leaves, for every row and 96 columns of it, the largest stored value and the sum of the exponentials
// relative to that one, in parts [2 ceil(N / 192)][M]: the logits and what their loss needs.
template <bool BF16, bool EDGES>
__device__ __forceinline__ void two_run(const uint8_t* __restrict__ a_codes, const uint8_t* __restrict__ a_scales, const uint8_t* __restrict__ b_codes,
                                        const uint8_t* __restrict__ b_scales, int M, int N, int K, float alpha, uint16_t* __restrict__ c, int late,
                                        [[maybe_unused]] float2* __restrict__ parts) {
    extern __shared__ uint32_t smem[];
    uint8_t* lds = reinterpret_cast<uint8_t*>(smem);
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)smem;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wm = wave >> 1, wn = wave & 1;
    const int nk = BF16 ? K / 32 : K / kBK, groups = K / 32;
    const int tiles_m = (M + kTwoM - 1) / kTwoM, tiles_n = (N + kTwoN - 1) / kTwoN, tiles = tiles_m * tiles_n;
    const int64_t block_row = (int64_t)nk * 1024;   // 16 rows of codes
    const int b_unit = wave < 3 ? wave : 2;         // of B's scale rows, 64 at a time: the fourth wave repeats the third's request

    // the second workgroup of a CU starts `late` x 1024 cycles late, so that the two do not reach their epilogues together (16384 x 4608 x
    // 1536 64.8 -> 64.1 us; 12 of them instead of 4 lose 5)
    if ((int)blockIdx.x >= (int)gridDim.x / 2)
        for (int i = 0; i < late; ++i) __builtin_amdgcn_s_sleep(16);

    // The tile that requests go to, its panels and this lane's place in them
    int m0, n0;
    [[maybe_unused]] int tile_n;
    const uint8_t *pa[4], *pb[3], *psa, *psb;
    uint32_t in_block, lane_sa, lane_sb;
    // scales of the four K steps from ks on; a short last block takes the row's final 16 bytes
    const auto scales_at = [&](int ks) { return ks + 4 <= nk ? ks : nk - 4; };
    const auto request_scales = [&](int ks) {
        const int at = scales_at(ks) * 4;
        const uint32_t to = lds_base + kTwoScales + ((ks >> 2) & 1) * kTwoScaleBuf;
        load_lds_b128_s(psa + at, lane_sa, to + wave * 1024);
        load_lds_b128_s(psb + at, lane_sb, to + kTwoM * 16 + b_unit * 1024);
    };
    const auto begin = [&](int t) {   // its first K step is on its way behind this
        int lane = (int)threadIdx.x & 63, tm, tn;
        asm volatile("" : "+v"(lane));
        tile_of_run<4>(xcd_run(t, tiles), tiles_m, tiles_n, tm, tn);
        m0 = tm * kTwoM;
        n0 = tn * kTwoN;
        tile_n = tn;
        // in a 1 KiB block of 16 rows: the 16 bytes that belong at lane * 16 of its LDS image
        in_block = (lane >> 2) * 64 + ((lane & 3) ^ ((lane >> 4) & 3)) * 16;
        const auto block_at = [&](const uint8_t* codes, int b, int rows) {   // 16-row block b, the last one past the end
            if (EDGES) b = b < (rows - 1) >> 4 ? b : (rows - 1) >> 4;
            return codes + b * block_row;
        };
#pragma unroll
        for (int j = 0; j < 4; ++j) pa[j] = block_at(a_codes, m0 / 16 + wave * 4 + j, M) - 1024 * j;
#pragma unroll
        for (int j = 0; j < 3; ++j) pb[j] = block_at(b_codes, n0 / 16 + wave * 3 + j, N) - 1024 * j;
        if constexpr (!BF16) {
            psa = a_scales + (int64_t)m0 * groups;
            psb = b_scales + (int64_t)n0 * groups;
            int ra = wave * 64 + lane, rb = b_unit * 64 + lane;
            if (EDGES) {
                ra = ra < M - 1 - m0 ? ra : M - 1 - m0;
                rb = rb < N - 1 - n0 ? rb : N - 1 - n0;
            } else {
                psa += (int64_t)wave * 64 * groups;
                psb += (int64_t)b_unit * 64 * groups;
                ra = rb = lane;
            }
            lane_sa = (uint32_t)(ra * groups);
            lane_sb = (uint32_t)(rb * groups);
            request_scales(0);
        }
        two_lds_base(lds_base + wave * 4096);
        two_request<0>(pa[0], in_block);
        two_request<1>(pa[1], in_block);
        two_request<2>(pa[2], in_block);
        two_request<3>(pa[3], in_block);
        two_lds_base(lds_base + kTwoBOff + wave * 3072);
        two_request<0>(pb[0], in_block);
        two_request<1>(pb[1], in_block);
        two_request<2>(pb[2], in_block);
    };
    int t = (int)blockIdx.x;
    if (t >= tiles) return;
    begin(t);
    for (bool first_tile = true;; first_tile = false) {
        int lane = (int)threadIdx.x & 63;
        asm volatile("" : "+v"(lane));   // worked out per tile: held through the epilogue these values would not fit
        const int lrow = lane & 31, half = lane >> 5;
        // this lane's 16 bytes of its wave's first A rows, in either half of a K step.  A wave's columns are 64 wn .. + 63 and 128 + 32 wn ..
        // + 31 of the tile, so that two of its blocks make whole lines of the result.
        const int swz = (lrow >> 2) & 3;
        // (a lane's eight bf16 of an instruction are piece half of the row's four, then piece 2 + half)
        const uint32_t a_off0 = (wm * 128 + lrow) * kRowBytes + ((BF16 ? half : 2 * half) ^ swz) * 16;
        const uint32_t a_off1 = (wm * 128 + lrow) * kRowBytes + ((BF16 ? 2 + half : 2 * half + 1) ^ swz) * 16;
        const int to_b = kTwoBOff + (wn * 64 - wm * 128) * kRowBytes, to_b2 = kTwoBOff + (128 + wn * 32 - wm * 128) * kRowBytes;   // uniform
        const uint32_t sc_off = (wm * 128 + lrow) * 16 + half * 2;   // the two scale bytes of this lane's half
        v16f acc[kTwoTM][kTwoTN];

        // One K step of slot ks % 2: its requests have had the step before to arrive; those of the next step, into the other slot, go out among
        // the first half's products.  Higher priority while it has products to issue: the CU's other workgroup, which waits or is
        // about to, gives way (16384 x 4608 x 8192 on zero codes 208 -> 193 us, 16384 x 1536 x 4096 51.6 -> 49.8).
        const auto step = [&](auto first_tag, int ks) {
            constexpr bool FIRST = decltype(first_tag)::value;
            const int slot = ks & 1;
            // a tile's first step is older than the stores of the tile before: 24 a wave, all of them where there are no edges
            if (FIRST && !EDGES && !first_tile) __builtin_amdgcn_s_waitcnt(vmcnt_imm(24));
            else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
            const int next = ks + 1 < nk ? ks + 1 : nk - 1;   // past the end: a repeat that nobody reads
            const uint8_t* cur = lds + slot * kTwoSlot;
            const uint32_t to = lds_base + (slot ^ 1) * kTwoSlot;
            uint32_t sca[kTwoTM], scb[kTwoTN];
            if constexpr (!BF16) {
                const uint8_t* sc = lds + kTwoScales + ((ks >> 2) & 1) * kTwoScaleBuf + (ks - scales_at(ks & ~3)) * 4 + sc_off;
                const uint8_t* sc_b = sc + kTwoM * 16 - wm * 2048;
#pragma unroll
                for (int i = 0; i < kTwoTM; ++i) sca[i] = *reinterpret_cast<const uint16_t*>(sc + i * 512);
                scb[0] = *reinterpret_cast<const uint16_t*>(sc_b + wn * 1024);
                scb[1] = *reinterpret_cast<const uint16_t*>(sc_b + wn * 1024 + 512);
                scb[2] = *reinterpret_cast<const uint16_t*>(sc_b + 2048 + wn * 512);
            }
            const uint8_t* c0 = cur + a_off0;
            const uint8_t* c1 = cur + a_off1;
            __builtin_amdgcn_s_setprio(2);
            uint4 a[kTwoTM], b[kTwoTN], b1[kTwoTN];
            b[0] = *reinterpret_cast<const uint4*>(c0 + to_b);
            b[1] = *reinterpret_cast<const uint4*>(c0 + to_b + 2048);
            b[2] = *reinterpret_cast<const uint4*>(c0 + to_b2);
#pragma unroll
            for (int i = 0; i < kTwoTM; ++i) a[i] = *reinterpret_cast<const uint4*>(c0 + i * 2048);
            __builtin_amdgcn_sched_barrier(0);
            // the next block's scales, behind the second step of a block, into the buffer that the block before has left
            if (!BF16 && (ks & 3) == 1 && ks + 3 < nk) request_scales(ks + 3);
            const auto products = [&](auto sub_tag, int i, const uint4 (&bb)[kTwoTN]) {
                constexpr int SUB = decltype(sub_tag)::value;
#pragma unroll
                for (int jj = 0; jj < kTwoTN; ++jj) {
                    const int j = i & 1 ? kTwoTN - 1 - jj : jj;   // back and forth, as in gemm.hip
                    v16f cin;
                    if constexpr (FIRST && SUB == 0) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) cin[e] = 0.0f;
                    } else {
                        cin = acc[i][j];
                    }
                    if constexpr (BF16) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, bb[j]), __builtin_bit_cast(v8bf, a[i]), cin, 0, 0, 0);
                    else acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(two_operand(bb[j]), two_operand(a[i]), cin, 4, 4, SUB, (int)scb[j], SUB, (int)sca[i]);
                }
            };
#pragma unroll
            for (int i = 0; i < kTwoTM; ++i) {
                if (i == 0) b1[0] = *reinterpret_cast<const uint4*>(c1 + to_b);
                if (i == 1) b1[1] = *reinterpret_cast<const uint4*>(c1 + to_b + 2048);
                if (i == 2) b1[2] = *reinterpret_cast<const uint4*>(c1 + to_b2);
                if (i == 0) {
                    two_lds_base(to + wave * 4096);
                    two_request<0>(pa[0] + next * 1024, in_block);
                    two_request<1>(pa[1] + next * 1024, in_block);
                }
                if (i == 1) {
                    two_request<2>(pa[2] + next * 1024, in_block);
                    two_request<3>(pa[3] + next * 1024, in_block);
                }
                if (i == 2) {
                    two_lds_base(to + kTwoBOff + wave * 3072);
                    two_request<0>(pb[0] + next * 1024, in_block);
                    two_request<1>(pb[1] + next * 1024, in_block);
                }
                if (i == 3) two_request<2>(pb[2] + next * 1024, in_block);
                products(std::integral_constant<int, 0>{}, i, b);
                a[i] = *reinterpret_cast<const uint4*>(c1 + i * 2048);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < kTwoTM; ++i) products(std::integral_constant<int, 1>{}, i, b1);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        };
        step(std::true_type{}, 0);
        for (int ks = 1; ks < nk; ++ks) step(std::false_type{}, ks);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        __syncthreads();

        // the next tile's first step, into the first slot; the result leaves through the second (26576 x 3008 x 1920 86.7 -> 84.5 us)
        const int row0 = m0, col0 = n0;
        [[maybe_unused]] const int segment = 2 * tile_n + wn;
        t += (int)gridDim.x;
        const bool more = t < tiles;
        if (more) begin(t);

        // bf16 through 4 KiB per wave: 32 rows of the wave's first two blocks of columns, then 64 rows of its third
        int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(ln));   // what is worked out from it stays behind the K loop
        uint8_t* region = lds + kTwoSlot + wave * 4096;
        const int chunk = ln & 7, rsub = ln >> 3;
        uint8_t* wr = region + (ln & 31) * 128 + (ln >> 5) * 8;
        const int wsw = (ln & 7) * 16;
        const uint8_t* rd = region + rsub * 128 + ((chunk ^ rsub) * 16);
        const int64_t pitch8 = (int64_t)N * 16;   // eight rows, in bytes
        const auto put_block = [&](v16f& v, int side) {   // BF16: leaves the rounded values in v
            const float f = BF16 ? 1.0f : alpha;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t p0 = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{v[4 * q] * f, v[4 * q + 1] * f}, v2bf));
                const uint32_t p1 = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{v[4 * q + 2] * f, v[4 * q + 3] * f}, v2bf));
                *reinterpret_cast<uint2*>(wr + (((side * 4 + q) * 16) ^ wsw)) = make_uint2(p0, p1);
                if constexpr (BF16) {
                    v[4 * q] = u2f(p0 << 16);
                    v[4 * q + 1] = u2f(p0 & 0xffff0000u);
                    v[4 * q + 2] = u2f(p1 << 16);
                    v[4 * q + 3] = u2f(p1 & 0xffff0000u);
                }
            }
        };
        const auto store_rows = [&](uint8_t* out, int row, bool col_ok) {   // of the lane's first row
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                typedef uint32_t u4v __attribute__((ext_vector_type(4)));
                const uint4 v = *reinterpret_cast<const uint4*>(rd + r * 1024);
                if (!EDGES || (col_ok && row + 8 * r < M)) __builtin_nontemporal_store(u4v{v.x, v.y, v.z, v.w}, reinterpret_cast<u4v*>(out + r * pitch8));
            }
        };
        {
            const int row = row0 + wm * 128 + rsub, col = col0 + wn * 64 + chunk * 8;
            uint8_t* out = reinterpret_cast<uint8_t*>(c + (int64_t)row * N + col);
#pragma unroll
            for (int i = 0; i < kTwoTM; ++i) {
                put_block(acc[i][0], 0);
                put_block(acc[i][1], 1);
                store_rows(out + i * 4 * pitch8, row + i * 32, col < N);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        {
            const int row = row0 + wm * 128 + rsub + (chunk >> 2) * 32, col = col0 + 128 + wn * 32 + (chunk & 3) * 8;
            uint8_t* out = reinterpret_cast<uint8_t*>(c + (int64_t)row * N + col);
#pragma unroll
            for (int i = 0; i < kTwoTM; i += 2) {
                put_block(acc[i][2], 0);
                put_block(acc[i + 1][2], 1);
                store_rows(out + i * 4 * pitch8, row + i * 32, col < N);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (BF16) {
            // a lane has 48 of its row's 96 columns (quads of them), the lane of the other half-wave the others
#pragma unroll
            for (int i = 0; i < kTwoTM; ++i) {
                if (EDGES) {
                    const int half_now = ln >> 5;
#pragma unroll
                    for (int j = 0; j < kTwoTN; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const bool in = col0 + (j < 2 ? wn * 64 + j * 32 : 128 + wn * 32) + 8 * q + 4 * half_now < N;   // N is a multiple of 8
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] = in ? acc[i][j][4 * q + e] : -INFINITY;
                        }
                }
                float top = -INFINITY;
#pragma unroll
                for (int j = 0; j < kTwoTN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) top = fmaxf(top, acc[i][j][e]);
                {
                    const auto r = __builtin_amdgcn_permlane32_swap(f2u(top), f2u(top), false, false);
                    top = fmaxf(u2f(r[0]), u2f(r[1]));
                }
                // Differences first: they are exact where a term counts, however large the logits are, and the largest element's term is one.  (With the
                // product top * log2 e, rounded, taken off in one fma, its rounding error is in every term: 3e-5 of a loss at logits of 1000, no finite one at 1e10.)
                const float ref = top == -INFINITY ? 0.0f : top;   // nothing but -inf: every term is zero
                float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < kTwoTN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) sum[e & 3] += __builtin_amdgcn_exp2f((acc[i][j][e] - ref) * kLog2e);
                float s = (sum[0] + sum[1]) + (sum[2] + sum[3]);
                {
                    const auto r = __builtin_amdgcn_permlane32_swap(f2u(s), f2u(s), false, false);
                    s = u2f(r[0]) + u2f(r[1]);
                }
                const int row = row0 + wm * 128 + i * 32 + (ln & 31);
                if (ln < 32 && (!EDGES || row < M)) parts[(int64_t)segment * M + row] = make_float2(top, s);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!more) break;
    }
}

template <bool EDGES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_mxfp4_tn_two_kernel(
    const uint8_t* __restrict__ a_codes, const uint8_t* __restrict__ a_scales, const uint8_t* __restrict__ b_codes, const uint8_t* __restrict__ b_scales,
    int M, int N, int K, float alpha, uint16_t* __restrict__ c, int late) {
    two_run<false, EDGES>(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, late, nullptr);
}
template <bool EDGES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_bf16_logits_kernel(
    const uint8_t* __restrict__ a, const uint8_t* __restrict__ b, int M, int N, int K, uint16_t* __restrict__ c, int late, float2* __restrict__ parts) {
    two_run<true, EDGES>(a, nullptr, b, nullptr, M, N, K, 1.0f, c, late, parts);
}

}  // namespace

bool gemm_two_serves(const TileProduct& p) {
    return p.a_tiled && p.b_tiled && !p.b_e5m2 && p.M > 0 && p.N >= 8 && p.N % 8 == 0 && p.K % kBK == 0 && p.K >= 4 * kBK && p.M < (1 << 30) && p.N < (1 << 30) &&
           p.K < (1 << 23) && (reinterpret_cast<uintptr_t>(p.c) & 15) == 0 &&
           ((reinterpret_cast<uintptr_t>(p.a_scales) | reinterpret_cast<uintptr_t>(p.b_scales)) & 3) == 0;
}
hipError_t gemm_two(const TileProduct& p, hipStream_t stream) {
    if (!gemm_two_serves(p) || p.mask) return hipErrorInvalidValue;
    const int tiles = ((p.M + kTwoM - 1) / kTwoM) * ((p.N + kTwoN - 1) / kTwoN);
    const auto go = [&](auto edges) {
        const auto kern = gemm_mxfp4_tn_two_kernel<decltype(edges)::value>;
        static std::atomic<bool> lds_allowed[kMaxDevices];
        const hipError_t e = allow_dynamic_lds(kern, kTwoLds, lds_allowed);
        if (e != hipSuccess) return e;
        // where a workgroup walks several tiles, a grid that is a multiple of eight: tile t and t + grid on the same XCD
        int grid = tiles < 2 * device_cus() ? tiles : 2 * device_cus();
        if (grid > 8 && grid < tiles) grid -= grid % 8;
        kern<<<dim3((unsigned)grid), dim3(256), kTwoLds, stream>>>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, p.M, p.N, p.K, p.alpha, static_cast<uint16_t*>(p.c),
                                                                     grid < tiles && p.K / kBK <= 16 ? 4 : 0);
        return hipGetLastError();
    };
    return p.M % kTwoM || p.N % kTwoN ? go(std::true_type{}) : go(std::false_type{});
}

// x [T, K], w [V, K] in blocks of 16 rows and 32 elements (see above), whole blocks of rows; logits 16-byte aligned
bool gemm_logits_serves(int64_t T, int64_t V, int64_t K) {
    return T > 0 && V >= 8 && V % 8 == 0 && K % 32 == 0 && K >= 64 && K <= 8192 && T < (1 << 24) && V < (1 << 24) && T * V < (1ll << 38) &&
           padded_rows(V) * K < (1ll << 35) - 2048;   // bf16_blocks' grid has an eighth as many threads, in whole workgroups, and fewer than 2^32
}
int64_t gemm_logits_segments(int64_t V) { return 2 * ((V + kTwoN - 1) / kTwoN); }
hipError_t gemm_logits(const void* x, const void* w, int64_t T, int64_t V, int64_t K, void* logits, void* parts, hipStream_t stream) {
    if (!gemm_logits_serves(T, V, K)) return hipErrorInvalidValue;
    const int64_t tiles = ((T + kTwoM - 1) / kTwoM) * ((V + kTwoN - 1) / kTwoN);
    const auto go = [&](auto edges) {
        const auto kern = gemm_bf16_logits_kernel<decltype(edges)::value>;
        static std::atomic<bool> lds_allowed[kMaxDevices];
        const hipError_t e = allow_dynamic_lds(kern, kTwoScales, lds_allowed);
        if (e != hipSuccess) return e;
        int64_t grid = tiles < 2 * device_cus() ? tiles : 2 * device_cus();
        if (grid > 8 && grid < tiles) grid -= grid % 8;
        kern<<<dim3((unsigned)grid), dim3(256), kTwoScales, stream>>>(static_cast<const uint8_t*>(x), static_cast<const uint8_t*>(w), (int)T, (int)V, (int)K,
                                                                      static_cast<uint16_t*>(logits), grid < tiles ? 8 : 0, static_cast<float2*>(parts));
        return hipGetLastError();
    };
    return T % kTwoM || V % kTwoN ? go(std::true_type{}) : go(std::false_type{});
}

}  // namespace qm
