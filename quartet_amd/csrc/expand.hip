// Packed MXFP4 [R, C] as the K x N operand of a product that contracts over its rows (the error-only scheme's Q(e) W and
// Q(e^T) x, backward.py:21-45).  The matrix instruction scales 32 consecutive contraction indices of a column together, but the
// tensor's E8M0 scales belong to 32 consecutive columns of a row, so codes cannot be multiplied as they are.  They can be
// widened: within a block of 32 rows and 32 columns every value is a code times a power of two, which six bits (E3M2: two
// mantissa bits where E2M1 has one) hold exactly as long as the row scales of the block lie within 5 octaves of the largest, and
// eight bits (E5M2) within 28.  The matrix instruction takes six bits at the rate of four, eight at half of it, and the bytes
// count too: the product of 4096^3 with its rotation runs 50 us with six and 63 with eight.  The format is chosen per block of 512 rows (four K
// steps) and 256 columns, by its scales alone (expand_formats.h); rows of zeros count for no range.  Rows of activations with
// outliers of three degrees of freedom stay within 5 octaves but for a block in a hundred or less.
//
// Output: slots of 2 KiB per 16 columns and 128 rows.  Eight bits: 16 columns x 64 rows (1 KiB, what one wave requests into
// LDS), twice.  Six bits: of every column's 24 bytes per 32 rows the first sixteen, [column][32 rows]; the last eight of
// 32 columns, [32 rows][column], lie in the second half of the even slot.  One E8M0 byte per column and 32 rows.  A block of 128
// x 128 that holds a value outside the range says so in `lost`, and the columns it touches are computed once more from the packed
// tensors (ExactJob): results never depend on the spread of the scales.
//
// Bound by memory: half a byte read and three quarters (or one) written per element; 14.3 us for 4096 x 4096 twice in either format
// (12.9 where only eight bits exist: packing six bits and the look at the format cost more than the bytes saved).  A thread takes
// four consecutive rows and 16 columns;
// v_perm_b32 looks four codes at a time up in an eight-byte table of the row's E5M2 magnitudes, eight more turn 4 x 4 bytes
// round, and the transposed dwords meet in LDS.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "expand_formats.h"
#include "qm_jobs.h"
#include "qm_kernels.h"
#include "qm_math.h"

namespace qm {

namespace {

constexpr int kTile = 128;                       // rows and columns per workgroup
constexpr int kColPitch = 128, kGroupPad = 32;   // LDS: 128 bytes per column, 16 columns padded by 32 bytes (banks)
constexpr int kTop = 13, kBias = 15;             // E5M2: the largest code, 6 = 1.5 * 2^2, times 2^13 is the largest value used, 1.5 * 2^15

// the E5M2 or E3M2 magnitude bits of the codes 0 .. 7 times 2^(x - bias), x >= 0; x < 0: zeros
__device__ __forceinline__ void magnitude_table(int x, uint32_t& lo, uint32_t& hi) {
    // x >= 2: code 1 (0.5) has the exponent field x - 1, codes 2, 3 (1, 1.5) x, 4, 5 x + 1, 6, 7 x + 2; odd codes mantissa 10
    const uint32_t e = 4u * (uint32_t)x;
    lo = ((e - 4u) << 8) | (e << 16) | ((e | 2u) << 24);
    hi = (e + 4u) | ((e + 6u) << 8) | ((e + 8u) << 16) | ((e + 10u) << 24);
    if (x == 1) lo = 0x06040200u;                             // 0.5 * 2^-14 is subnormal
    if (x == 0) { lo = 0x03020100u; hi = 0x0a080604u; }       // 0.5, 1, 1.5 times 2^-15 are
    if (x < 0) lo = hi = 0u;
}

struct ExpandJob {
    static constexpr int kLds = kTile * kColPitch + (kTile / 16) * kGroupPad + kTile * 4 + 16;
    static constexpr int kWaves = 1;
    E5m2Args a;
    unsigned grid_r, blocks;
    explicit ExpandJob(const E5m2Args& args)
        : a(args), grid_r((unsigned)((args.R + kTile - 1) / kTile)), blocks((unsigned)(((args.R + kTile - 1) / kTile) * ((args.C + kTile - 1) / kTile))) {}

    __device__ __forceinline__ void run(unsigned bid) const {
        uint8_t* turned = reinterpret_cast<uint8_t*>(job_lds);
        uint32_t* row_scales = reinterpret_cast<uint32_t*>(turned + kTile * kColPitch + (kTile / 16) * kGroupPad);   // [128 rows], a byte per 32 columns
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const unsigned bc = bid / grid_r, br = bid - bc * grid_r;
        const int r0 = (int)br * kTile, c0 = (int)bc * kTile;
        const int R = (int)a.R, C = (int)a.C, csteps = (int)(padded_cols(C) / 128), ksteps = (int)(padded_cols(R) / 128);
        if (tid < kTile) row_scales[tid] = r0 + tid < R ? *reinterpret_cast<const uint32_t*>(a.scales_in + (int64_t)(r0 + tid) * csteps * 4 + bc * 4) : 0u;
        // rows r .. r + 3 (all inside or all outside: R is a multiple of 32), columns 16 g .. 16 g + 15
        const int g = lane & 7, quad = wave * 8 + (lane >> 3), r = r0 + 4 * quad;
        uint2 codes[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            codes[i] = make_uint2(0u, 0u);
            if (r < R) codes[i] = *reinterpret_cast<const uint2*>(a.codes_in + tiled_code_offset(r + i, bc, csteps) + g * 8);
        }
        job_requests_issued();
        const bool six = a.wide && a.wide[(int64_t)(bc / 2) * ((ksteps + 3) / 4) + br / 4] == 0;
        __syncthreads();
        const int top_octaves = six ? kTop6 : kTop, bias = six ? kBias6 : kBias, even_sign = six ? 2 : 4, odd_sign = six ? 2 : 0;
        // per 32 rows the largest scale of each column group: a wave's quads lie in one block of 32 rows
        uint32_t top = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t s = (row_scales[wave * 32 + i * 4 + (lane >> 4)] >> (8 * (g >> 1))) & 0xffu;
            top = s > top ? s : top;
        }
        top = max(top, (uint32_t)__shfl_xor((int)top, 16, 64));
        top = max(top, (uint32_t)__shfl_xor((int)top, 32, 64));
        const int block_scale = top == 255u ? 255 : (int)top - ((int)top < top_octaves ? (int)top : top_octaves);
        bool lost = false;
        uint32_t even[4][2], odd[4][2];   // row i: bytes of columns 8 h + 0, 2, 4, 6 and 8 h + 1, 3, 5, 7
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int x = bias + (int)((row_scales[4 * quad + i] >> (8 * (g >> 1))) & 0xffu) - block_scale;
            uint32_t lo, hi;
            magnitude_table(x, lo, hi);
            lost |= x < 0 && top != 255u && ((codes[i].x | codes[i].y) & 0x77777777u);   // a NaN scale: the block is NaN as it is
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t w = h ? codes[i].y : codes[i].x;
                even[i][h] = __builtin_amdgcn_perm(hi, lo, w & 0x07070707u) | ((w & 0x08080808u) << even_sign);
                odd[i][h] = __builtin_amdgcn_perm(hi, lo, (w >> 4) & 0x07070707u) | ((w & 0x80808080u) >> odd_sign);
            }
        }
        // 4 rows x 4 columns of bytes turned round: dword = the four rows of one column
        uint8_t* dst = turned + g * (16 * kColPitch + kGroupPad) + quad * 4;
        const auto turn = [&](const uint32_t (&m)[4][2], int h, int first) {
            const uint32_t p01a = __builtin_amdgcn_perm(m[1][h], m[0][h], 0x05010400u), p01b = __builtin_amdgcn_perm(m[1][h], m[0][h], 0x07030602u);
            const uint32_t p23a = __builtin_amdgcn_perm(m[3][h], m[2][h], 0x05010400u), p23b = __builtin_amdgcn_perm(m[3][h], m[2][h], 0x07030602u);
            const uint32_t col[4] = {__builtin_amdgcn_perm(p23a, p01a, 0x05040100u), __builtin_amdgcn_perm(p23a, p01a, 0x07060302u),
                                     __builtin_amdgcn_perm(p23b, p01b, 0x05040100u), __builtin_amdgcn_perm(p23b, p01b, 0x07060302u)};
#pragma unroll
            for (int j = 0; j < 4; ++j) *reinterpret_cast<uint32_t*>(dst + (8 * h + first + 2 * j) * kColPitch) = col[j];
        };
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            turn(even, h, 0);
            turn(odd, h, 1);
        }
        // the block's scale byte of this wave's 32 rows, one per column group of 32, at [column group][wave]
        const bool any_lost = __syncthreads_or(lost);
        uint8_t* group_scales = reinterpret_cast<uint8_t*>(row_scales);   // everyone has read the row scales
        if (lane < 8 && !(lane & 1)) group_scales[(lane >> 1) * 4 + wave] = (uint8_t)block_scale;
        __syncthreads();
        job_stores_next();
        const int col = lane >> 2, rows32 = lane & 3;
#pragma unroll
        for (int it = 0; it < 2 && six; ++it) {   // 16 columns, 32 rows of one to a lane: 24 bytes, sixteen of them and eight apart
            const int cg = it * 4 + wave;
            if (c0 + cg * 16 < C) {
                const uint4* src = reinterpret_cast<const uint4*>(turned + cg * (16 * kColPitch + kGroupPad) + col * kColPitch + rows32 * 32);
                const uint4 v0 = src[0], v1 = src[1];
                const auto pack = [](uint32_t v) { return __builtin_amdgcn_udot4(v, 0x4001u, 0u, false) | (__builtin_amdgcn_udot4(v, 0x40010000u, 0u, false) << 12); };
                const uint32_t w0 = pack(v0.x), w1 = pack(v0.y), w2 = pack(v0.z), w3 = pack(v0.w), w4 = pack(v1.x), w5 = pack(v1.y), w6 = pack(v1.z), w7 = pack(v1.w);
                uint8_t* panel = a.values + (((int64_t)(c0 / 16 + cg) * ksteps + br) << 11);
                *reinterpret_cast<uint4*>(panel + lane * 16) = make_uint4(w0 | (w1 << 24), (w1 >> 8) | (w2 << 16), (w2 >> 16) | (w3 << 8), w4 | (w5 << 24));
                uint8_t* pair = a.values + (((int64_t)((c0 / 16 + cg) & ~1) * ksteps + br) << 11);
                *reinterpret_cast<uint2*>(pair + 1024 + rows32 * 256 + ((cg & 1) * 16 + col) * 8) = make_uint2((w5 >> 8) | (w6 << 16), (w6 >> 16) | (w7 << 8));
            }
        }
        // eight bits: blocks of 16 columns x 64 rows, 1 KiB each; a wave writes one at a time
#pragma unroll
        for (int it = 0; it < 4 && !six; ++it) {
            const int block = it * 4 + wave, cg = block >> 1, half = block & 1;   // 16 blocks of the workgroup
            if (c0 + cg * 16 < C) {
                const uint4 v = *reinterpret_cast<const uint4*>(turned + cg * (16 * kColPitch + kGroupPad) + (lane >> 2) * kColPitch + half * 64 + (lane & 3) * 16);
                *reinterpret_cast<uint4*>(a.values + (((int64_t)(c0 / 16 + cg) * ksteps + br) << 11) + half * 1024 + lane * 16) = v;
            }
        }
        if (tid < kTile && c0 + tid < C)
            *reinterpret_cast<uint32_t*>(a.scales + (int64_t)(c0 + tid) * ksteps * 4 + br * 4) = *reinterpret_cast<const uint32_t*>(group_scales + (tid >> 5) * 4);
        if (tid == 0) a.lost[(int64_t)bc * ksteps + br] = any_lost ? 1 : 0;
    }
};

// One value of a packed tensor (tiled codes)
__device__ __forceinline__ float packed_value(const uint8_t* codes, const uint8_t* scales, int64_t r, int c, int ksteps) {
    const uint32_t s = scales[r * ksteps * 4 + c / 32];
    const uint32_t q = codes[tiled_code_offset(r, c / 128, ksteps) + (c & 127) / 2] >> (4 * (c & 1));
    const uint32_t m = q & 7u;
    const float v = m < 2 ? 0.5f * (float)m : u2f(((m >> 1) + 126u) << 23) * ((m & 1) ? 1.5f : 1.0f);
    const float scale = s == 255u ? __builtin_nanf("") : s ? u2f(s << 23) : u2f(1u << 22);
    return ((q & 8u) ? -v : v) * scale;
}

// A workgroup looks at one panel of 128 columns of one product and, should a block of it have lost values, computes the
// panel's share of rows, two at a time, sum by sum.  It takes two microseconds to find nothing (4096 x 4096 x 4096), and
// scales of one column group spread over more than 2^28 within 32 rows to make it find something.
constexpr int kShares = 4;
struct ExactJob {
    static constexpr int kLds = 256 * 4;
    static constexpr int kWaves = 1;
    E5m2Exact p;
    unsigned blocks;
    explicit ExactJob(const E5m2Exact& e) : p(e), blocks((unsigned)((e.b.C + kTile - 1) / kTile) * kShares) {}

    __device__ __forceinline__ void run(unsigned bid) const {
        const int tid = threadIdx.x;
        const int panel = (int)(bid / kShares), share = (int)(bid % kShares);
        const int R = (int)p.b.R, C = (int)p.b.C, ksteps = (int)(padded_cols(R) / 128), csteps = (int)(padded_cols(C) / 128);
        uint32_t lost = 0;
        for (int i = tid; i < ksteps; i += 256) lost |= p.b.lost[(int64_t)panel * ksteps + i];
        if (!__syncthreads_or((int)lost)) return;
        float* row = reinterpret_cast<float*>(job_lds) + (tid & 128);
        const int j = tid & 127, n = panel * 128 + j, block = j & ~(p.hd - 1), in_block = j & (p.hd - 1);
        for (int64_t m0 = 2 * share; m0 < p.M; m0 += 2 * kShares) {
            const int64_t m = m0 + (tid >> 7);
            const bool inside = m < p.M && n < C;
            float sum = 0.0f;
            if (inside)
                for (int k = 0; k < R; ++k)
                    sum += packed_value(p.a_codes, p.a_scales, m, k, ksteps) * packed_value(p.b.codes_in, p.b.scales_in, k, n, csteps);
            float v = bf16_to_f32(f32_to_bf16(sum * p.alpha));
            if (inside) {
                const uint32_t keep = (p.mask[m * (C / 8) + n / 8] >> (n & 7)) & 1u;
                const uint32_t words[4] = {p.signs.w[0], p.signs.w[1], p.signs.w[2], p.signs.w[3]};
                uint32_t word = words[0];
#pragma unroll
                for (int w = 1; w < 4; ++w) word = in_block / 32 == w ? words[w] : word;
                v *= keep ? 1.0f : 0.0f;
                if ((word >> (in_block & 31)) & 1u) v = -v;
            }
            __syncthreads();
            row[j] = v;
            __syncthreads();
            float turned = 0.0f;
            for (int i = 0; i < p.hd; ++i) turned += (__popc(i & in_block) & 1) ? -row[block + i] : row[block + i];
            const uint16_t o = f32_to_bf16(turned * p.rot_c);
            if (inside) {
                if (p.out_dtype == BF16) reinterpret_cast<uint16_t*>(p.c)[m * C + n] = o;
                else reinterpret_cast<float*>(p.c)[m * C + n] = bf16_to_f32(o);
            }
        }
    }
};

}  // namespace

hipError_t e5m2_exact_pair(const E5m2Exact& a, const E5m2Exact& b, hipStream_t stream) {
    launch_jobs(stream, ExactJob(a), ExactJob(b));
    return hipGetLastError();
}

hipError_t expand_e5m2_pair(const E5m2Args& a, const E5m2Args& b, hipStream_t stream) {
    launch_jobs(stream, ExpandJob(a), ExpandJob(b));
    return hipGetLastError();
}

}  // namespace qm
