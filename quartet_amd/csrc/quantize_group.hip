// Fast path of the fused block-Hadamard + MXFP4 quantizer ("group layout"): Hadamard block 32 for row-major,
// transposed and packed (re-quantize) input; Hadamard blocks 64 and 128 for row-major input.
//
// Same arithmetic as quantize.hip (the reference kernel
// src/models/quantization/quantizers/mxfp4_triton.py:19-174), different work decomposition: one lane
// owns a whole MX group of 32 values in registers, so
//   - the five butterfly stages, the group statistics and the scale are computed without any
//     cross-lane traffic and the per-group scalar work (sqrt, exponent extraction) is done once
//     instead of once per quarter group;
//   - the column sign of rotated element j is the same for every lane (j is a register index), so it
//     folds into the multiply by hd^-1/2;
//   - rounding, sign and nibble packing are done by gfx950's FP4 converts:
//       RTN  v_cvt_scalef32_pk_fp4_f32 is round-to-nearest-even; the reference rounds ties toward
//            zero, which differs exactly at .75, 1.75, 3.5: below_ties() (qm_math.h) moves those three below themselves
//            in one fused multiply-add.
//       SR   v_cvt_scalef32_sr_pk_fp4_f32 rounds up iff floor(p * 2^22) + R >= 2^22 with p the position
//            inside the bracket and R = bits 31..10 of the random operand for the pair's first element,
//            bits 30..9 for its second (measured).  With R = the element's 22-bit field of the Philox stream this is
//            "u < p" for the uniform that stream defines (qm_math.h), bit for bit.  Each element gets its
//            own field (two converts per pair, merged with one mask).
//     The reference's sign rule "negative unless t > 0" makes +0 negative.  The rotation therefore hands out the negated
//     group (its factor is -hd^-1/2), on which the rule is "positive unless n < 0": zeros arrive at the converts as +0,
//     and one XOR gives eight codes their signs.
// Issue cost on the vector unit with several waves on a SIMD (measured): fp32 add / multiply / fma and logic 2.5 to 2.7 cycles
// per wave instruction, shifts, compares, selects, permutes and min/max 4.3, 64-bit multiply-add 4.6, FP4 -> fp32 convert 4.6,
// fp32 -> FP4 convert of a pair 9, with stochastic rounding 13.  Per group of 32: RTN about 1250 cycles, 1580 before the two
// forms above and the mask bits by subtraction; SR about 1470, 1600 before.
// Outputs are one 16-byte code store, one scale byte and one mask dword per lane, all contiguous across
// lanes; the input is read as 64 (bf16) or 128 (fp32) contiguous bytes per lane.
// The tiled row-major, transposed and re-quantizing kernels are written as jobs (qm_jobs.h) so that the whole-layer
// entry points can issue two of them in one grid.  rotate = false (row-major kernel only) skips the butterfly: the
// caller has already applied a dense rotation.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "expand_formats.h"
#include "hadamard_octet.h"
#include "lds_requests.h"
#include "qm_jobs.h"
#include "qm_kernels.h"
#include "qm_math.h"
#include "streaming.h"
#include "quantize_group.h"

namespace qm {

namespace {

// what the lanes of a wave wrote to LDS before is read by its other lanes behind
__device__ __forceinline__ void wave_settle() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- dense 32x32 rotation (rerotate="O32", quantizers/mxfp4.py:61-64 of the reference) on the matrix pipe ----------
// The reference applies the matrix with tl.dot inside its kernel (mxfp4_triton.py:44-45).  Here each lane owns one
// group of 32 values; v_mfma_f32_32x32x2_f32 computes D[j][n] += H[k][j] x[n][k] for 32 groups n at a time, and sixteen
// chained instructions walk k = 0..31.  The instruction evaluates acc = fma(a, b, acc) per term in ascending k
// (measured against every candidate order on random fp32 data: no mismatch), which is the order the test oracle states.
// Lanes 0..31 hold groups "lo", lanes 32..63 groups "hi": v_permlane32_swap deals a lane's pair (k, k+1) out as the two
// k rows the instruction wants from the two half-waves, and collects the results (a lane gets the 16 rotated values of
// its group that the other half-wave computed).  Every lane of the wave must be active.
typedef float v16f __attribute__((ext_vector_type(16)));
struct DenseFrag {
    float a[16];  // -H[2t + lane/32][lane%32], t = 0..15, H rounded to the tensor's dtype
};
__device__ __forceinline__ void load_dense_frag(const float* __restrict__ matrix, int dtype, DenseFrag& f) {
    const int lane = threadIdx.x & 63, j = lane & 31, half = lane >> 5;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float h = matrix[(2 * t + half) * 32 + j];
        if (dtype == BF16) h = bf16_to_f32(f32_to_bf16(h));
        f.a[t] = -h;   // negated, as quantize_group_regs takes the rotated group
    }
}
__device__ __forceinline__ void dense_rotate(float (&v)[32], const DenseFrag& f) {
    v16f lo, hi;
#pragma unroll
    for (int e = 0; e < 16; ++e) lo[e] = hi[e] = 0.0f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        // after the swap: first = (k = 2t of groups lo | k = 2t+1 of groups lo), second = the same of groups hi
        const auto r = __builtin_amdgcn_permlane32_swap(f2u(v[2 * t]), f2u(v[2 * t + 1]), false, false);
        lo = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[t], u2f(r[0]), lo, 0, 0, 0);
        hi = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[t], u2f(r[1]), hi, 0, 0, 0);
    }
    // accumulator element e of a lane is output row j = 8 (e / 4) + 4 (lane / 32) + e % 4 of group lane % 32
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const auto r = __builtin_amdgcn_permlane32_swap(f2u(lo[e]), f2u(hi[e]), false, false);
        v[8 * (e / 4) + (e % 4)] = u2f(r[0]);
        v[8 * (e / 4) + 4 + (e % 4)] = u2f(r[1]);
    }
}

// ---- Hadamard blocks 64 and 128 ---------------------------------------------------------------------------
// Same one-group-per-lane layout; a Hadamard chunk is HD/32 consecutive lanes (a lane pair or a quad).  The
// five in-register stages are followed by the stride-32 (and stride-64) stages across the lanes of the chunk, one
// DPP-fed multiply-add per element: own + partner in the lower lane of a butterfly, own - partner in the upper one.
// The upper lane's exact value is partner - own = -(own - partner): rounding is symmetric, so the negation commutes
// with it, and it is folded into the column sign applied at the end (a lane's values are negated once per stage in
// which it is the upper lane).  The column signs differ per lane of the chunk; they are applied as lane masks held in
// scalar registers (bit l of mask j: negate element j in lane l), one select per element.
template <int CTRL>
__device__ __forceinline__ void cross_lane_stage(float (&v)[32], float s) {
    // s = +1 in the lower lane, -1 in the upper one.  An instruction reads its own destination register from the
    // partner lane; the leading s_nop keeps the two wait states a DPP read needs after a vector write to that register
    // (the compiler does not look into assembly statements).
#define QM_X(N) "v_fmac_f32_dpp %" #N ", %" #N ", %16 quad_perm:[%17,%18,%19,%20] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define QM_STAGE16(B)                                                                                                   \
    asm volatile("s_nop 1\n\t" QM_X(0) QM_X(1) QM_X(2) QM_X(3) QM_X(4) QM_X(5) QM_X(6) QM_X(7) QM_X(8) QM_X(9) QM_X(10) QM_X(11)  \
                 QM_X(12) QM_X(13) QM_X(14) QM_X(15)                                                                     \
                 : "+v"(v[(B)]), "+v"(v[(B) + 1]), "+v"(v[(B) + 2]), "+v"(v[(B) + 3]), "+v"(v[(B) + 4]), "+v"(v[(B) + 5]),  \
                   "+v"(v[(B) + 6]), "+v"(v[(B) + 7]), "+v"(v[(B) + 8]), "+v"(v[(B) + 9]), "+v"(v[(B) + 10]),             \
                   "+v"(v[(B) + 11]), "+v"(v[(B) + 12]), "+v"(v[(B) + 13]), "+v"(v[(B) + 14]), "+v"(v[(B) + 15])          \
                 : "v"(s), "n"(CTRL & 3), "n"((CTRL >> 2) & 3), "n"((CTRL >> 4) & 3), "n"((CTRL >> 6) & 3))
    QM_STAGE16(0);
    QM_STAGE16(16);
#undef QM_STAGE16
#undef QM_X
}

// Per-element negation fields of the wide kernel: bit p of field j = column sign of rotated element 32 p + j, xor 1 for
// the lanes of a chunk whose index has an odd number of set bits (their values come out of the cross-lane stages negated).
template <int HD>
SignBits wide_sign_fields(const SignBits& sb) {
    constexpr int P = HD / 32;
    SignBits sf{{0u, 0u, 0u, 0u}};
    for (int j = 0; j < 32; ++j) {
        uint32_t field = 0u;
        for (int p = 0; p < P; ++p) field |= (((sb.w[p] >> j) & 1u) ^ (uint32_t)(__builtin_popcount((unsigned)p) & 1)) << p;
        sf.w[(j * P) >> 5] |= field << ((j * P) & 31);
    }
    return sf;
}


// What a quantizer's rotation needs at run time: the factor hd^-1/2 and its column signs (HD = 32: one word; wider blocks:
// the per-element fields of wide_sign_fields)
struct Rotation {
    float c;
    SignBits signs;
};
template <int HD>
Rotation make_rotation(int dtype, const SignBits& sb) {
    if constexpr (HD == 32) return Rotation{hadamard_scale(32, dtype), sb};
    else return Rotation{hadamard_scale(HD, dtype), wide_sign_fields<HD>(sb)};
}
// -(x @ H) for a lane's group of 32; a block of 64 or 128 spans the lane pair or quad whose lanes hold its groups in order
template <int HD>
__device__ __forceinline__ void rotate_block(float (&v)[32], const Rotation& r) {
    if constexpr (HD == 32) {
        rotate_group(v, r.c, r.signs.w[0]);
    } else {
        butterfly32(v);
        const int part = (int)threadIdx.x & (HD / 32 - 1);
        cross_lane_stage<0xB1>(v, (part & 1) ? -1.0f : 1.0f);                           // quad_perm [1,0,3,2]: stride 32
        if constexpr (HD == 128) cross_lane_stage<0x4E>(v, (part & 2) ? -1.0f : 1.0f);  // quad_perm [2,3,0,1]: stride 64
        // the fields hold, per element j, HD/32 bits: bit p = negate element j in the chunk's lane p (column sign xor the
        // stage negations above).  field * 0x5555... (or 0x1111...) spreads it over the wave's chunks.
        constexpr int P = HD / 32;
        constexpr uint32_t kUnit = P == 2 ? 0x55555555u : 0x11111111u;
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const uint32_t field = (r.signs.w[(j * P) >> 5] >> ((j * P) & 31)) & ((1u << P) - 1u);  // wave-uniform: scalar registers
            const uint32_t half = field * kUnit;
            const uint64_t m = ((uint64_t)half << 32) | half;
            const float scaled = v[j] * -r.c;
            asm("v_cndmask_b32_e64 %0, %1, -%1, %2" : "=v"(v[j]) : "v"(scaled), "s"(m));
        }
    }
}

// rotate (hd = 32) + quantize the group in v; gi is its logical (row-major) group index, which also keys the
// random stream; ci is the index of its 16 code bytes in the code buffer (= gi for row-major codes)
template <typename T, int MODE, bool WANT_MASK>
__device__ __forceinline__ void finish_group(float (&v)[32], int64_t gi, int64_t ci, float c, uint32_t sign_word,
                                             uint64_t seed, const GroupOut& out, bool rotate) {
    rotate_group(v, c, sign_word, rotate);
    GroupCodes o;
    quantize_group_regs<MODE, WANT_MASK>(v, seed, gi, o);
    out.codes[ci] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
    out.scales[gi] = (uint8_t)o.scale_byte;
    if constexpr (WANT_MASK) out.maskbits[gi] = o.keep;
    if (out.dequant) store_dequant<T>(reinterpret_cast<T*>(out.dequant) + gi * 32, o);
}

template <typename T, int MODE, bool WANT_MASK>
__global__ __launch_bounds__(256) void quantize_rowmajor_g32_kernel(const T* __restrict__ x, int64_t n_groups, float c,
                                                                    uint32_t sign_word, uint64_t seed, GroupOut out,
                                                                    int rotate) {
    job_starts();
    const int64_t gi = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gi >= n_groups) return;
    float v[32];
    load_group<T>(x + gi * 32, v);
    job_requests_issued();
    finish_group<T, MODE, WANT_MASK>(v, gi, gi, c, sign_word, seed, out, rotate != 0);
}

// Row-major input with a dense rotation: one group per lane, flat over the tensor; row-major or tiled code bytes.
template <typename T, int MODE, bool WANT_MASK>
__global__ __launch_bounds__(256) void quantize_rowmajor_dense_kernel(const T* __restrict__ x, int64_t n_groups, int groups_per_row,
                                                                      const float* __restrict__ matrix, uint64_t seed,
                                                                      GroupOut out, int tiled) {
    const int64_t gi = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool valid = gi < n_groups;
    DenseFrag frag;
    load_dense_frag(matrix, sizeof(T) == 2 ? BF16 : F32, frag);
    float v[32];
    if (valid) {
        load_group<T>(x + gi * 32, v);
    } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) v[i] = 0.0f;
    }
    dense_rotate(v, frag);  // the whole wave, also past the end of the tensor
    if (!valid) return;
    GroupCodes o;
    quantize_group_regs<MODE, WANT_MASK>(v, seed, gi, o);
    int64_t ci = gi;
    if (tiled) {
        const int64_t row = gi / groups_per_row;
        const int g = (int)(gi - row * groups_per_row);
        ci = (row >> 4) * 16 * groups_per_row + ((g >> 2) * 64 + (int)(row & 15) * 4 + (g & 3));
    }
    out.codes[ci] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
    out.scales[gi] = (uint8_t)o.scale_byte;
    if constexpr (WANT_MASK) out.maskbits[gi] = o.keep;
    if (out.dequant) store_dequant<T>(reinterpret_cast<T*>(out.dequant) + gi * 32, o);
}

template <typename T, bool WANT_MASK>
void launch_rowmajor_dense(int mode, const void* x, int64_t rows, int64_t cols, const float* matrix, uint64_t seed,
                           const GroupOut& out, bool tiled, hipStream_t stream) {
    const T* xp = reinterpret_cast<const T*>(x);
    const int64_t n_groups = rows * cols / 32;
    const int gpr = (int)(cols / 32);
    dim3 grid((unsigned)((n_groups + 255) / 256)), block(256);
    switch (mode) {
        case QUEST_RTN: quantize_rowmajor_dense_kernel<T, QUEST_RTN, WANT_MASK><<<grid, block, 0, stream>>>(xp, n_groups, gpr, matrix, seed, out, (int)tiled); break;
        case ABSMAX_RTN: quantize_rowmajor_dense_kernel<T, ABSMAX_RTN, WANT_MASK><<<grid, block, 0, stream>>>(xp, n_groups, gpr, matrix, seed, out, (int)tiled); break;
        case ABSMAX_SR: quantize_rowmajor_dense_kernel<T, ABSMAX_SR, WANT_MASK><<<grid, block, 0, stream>>>(xp, n_groups, gpr, matrix, seed, out, (int)tiled); break;
        default: quantize_rowmajor_dense_kernel<T, QUEST_SR, WANT_MASK><<<grid, block, 0, stream>>>(xp, n_groups, gpr, matrix, seed, out, (int)tiled); break;
    }
}

// Waves on a SIMD that the grid of the backward pass's four quantizers (not the error signal's by themselves) is compiled for: as many as fit without scratch memory.  Left
// alone the compiler took 128 to 160 registers (three waves, four for whole tiles of blocks of 32) where 96 do for blocks of 32 and 107
// and 127 for blocks of 64 and 128; six waves would spill.  The other waves' arithmetic hides one's requests.  us of the grid, before
// and now: 1824 x 1408 x 2048 18.8 -> 14.5, 20000 x 704 x 704 33.8 -> 30.2, blocks of 64 8192 x 4096 x 4096 83.7 -> 76.3; per step
// 8192 x 4096 x 4096 279.4 -> 276.1, 8192 x 4096 x 11008 686.6 -> 682.7, blocks of 128 8192 x 1536 x 4608 185.5 -> 183.1.
constexpr int backward_waves(int hd) { return hd == 32 ? 5 : 4; }

// Tiled code layout ([rows/16][cols/128][16 rows][64 bytes]).  Workgroup b owns block b / chunks of 16 rows and run
// b % chunks of 512 columns (four code tiles); wave w owns rows 4w..4w+3 of the block, lane l its row l / 16 and
// group l % 16 of the run: the wave reads four contiguous KiB (bf16) and writes, per tile, four rows' 64-byte pieces
// = 256 contiguous bytes.  The four scale bytes of four adjacent groups are gathered into one dword store.
// A last run of one or two code tiles would leave three quarters or half of such a workgroup idle: its workgroups own 64 or 32 rows of that
// run instead, a lane per group.  us per training step with idle lanes and without: 16480 x 1728 x 640 111.6 -> 107.0, 24576 x 1152 x 640 113.7 -> 108.3,
// 16384 x 640 x 1920 115.5 -> 112.4; widths of whole runs the same.
// PADDED: any number of rows; columns that are not a multiple of 128 are completed with zero codes and scales.  (Whole tiles
// have instantiations of their own: the edge tests cost the kernel 5 to 10 %.)
template <typename T, int MODE, bool WANT_MASK, int HD = 32, bool PADDED = false>
struct RowmajorTiledJob {
    static constexpr int kLds = 0;
    static constexpr int kWaves = MODE == QUEST_RTN ? 8 : 0;   // forward: 62 registers; with padded extents 70 without the bound
    const T* x;
    int rows, groups, groups_p, chunks;   // groups of 32 per row: of the tensor, of its padded code tiles; runs of up to 16 in workgroups of 16 rows
    int narrow;                           // groups of the last run, 4 or 8, if it has workgroups of its own, or 0
    Rotation rot;
    uint64_t seed;
    const uint64_t* seed_base = nullptr;  // device memory, or null: a value the kernel adds to `seed` when it runs
    GroupOut out;
    unsigned wide_blocks, blocks;

    RowmajorTiledJob(const void* x_, int64_t rows_, int64_t cols_, const Rotation& rot_, uint64_t seed_, const GroupOut& out_)
        : x(reinterpret_cast<const T*>(x_)), rows((int)rows_), groups((int)(cols_ / 32)), groups_p((int)(padded_cols(cols_) / 32)),
          chunks((groups_p + 15) / 16), narrow(groups_p % 16 == 12 ? 0 : groups_p % 16), rot(rot_), seed(seed_), out(out_) {
        if (narrow) --chunks;
        wide_blocks = (unsigned)(padded_rows(rows_) / 16 * chunks);
        blocks = wide_blocks + (narrow ? (unsigned)((rows_ * narrow + 255) / 256) : 0u);
    }

    __device__ __forceinline__ void run(unsigned bid) const {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        unsigned rb;   // first block of 16 rows
        int g, rin;    // group within the row, row within the block
        const bool wide = bid < wide_blocks;
        if (wide) {
            rb = bid / (unsigned)chunks;
            g = (int)(bid - rb * chunks) * 16 + (lane & 15);
            rin = wave * 4 + (lane >> 4);
        } else {
            const int shift = narrow == 4 ? 2 : 3;
            rb = (bid - wide_blocks) << (narrow == 4 ? 2 : 1);
            g = chunks * 16 + ((int)threadIdx.x & (narrow - 1));
            rin = (int)threadIdx.x >> shift;
        }
        // groups_p is a multiple of four: quads of lanes leave together, but for the padding lanes of a row's last quad
        if (g >= (PADDED ? groups_p : groups)) return;
        if ((PADDED || !wide) && (int)rb * 16 + rin >= rows) return;
        // uniform 64-bit block bases + small per-lane offsets
        const int pitch = PADDED ? groups_p : groups;   // groups per row of the code and scale arrays
        const int64_t gi = (int64_t)rb * 16 * groups + (rin * groups + g);
        const int64_t ci = (int64_t)rb * 16 * pitch + ((rin >> 4) * 16 * pitch + (g >> 2) * 64 + (rin & 15) * 4 + (g & 3));
        if (PADDED && g >= groups) {
            out.codes[ci] = make_uint4(0u, 0u, 0u, 0u);
            return;
        }
        float v[32];
        load_group<T>(x + gi * 32, v);
        job_requests_issued();
        rotate_block<HD>(v, rot);
        GroupCodes o;
        quantize_group_regs<MODE, WANT_MASK>(v, seed_base ? seed + *seed_base : seed, gi, o);
        job_stores_next();
        out.codes[ci] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
        // quad_perm broadcasts of lanes 1, 2, 3 of each quad (0 from a padding lane: it has left)
        const uint32_t s1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o.scale_byte, 0x55, 0xf, 0xf, false);
        const uint32_t s2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o.scale_byte, 0xAA, 0xf, 0xf, false);
        const uint32_t s3 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o.scale_byte, 0xFF, 0xf, 0xf, false);
        if ((lane & 3) == 0) {
            const int64_t si = PADDED ? (int64_t)rb * 16 * pitch + (rin * pitch + g) : gi;
            *reinterpret_cast<uint32_t*>(out.scales + si) = o.scale_byte | (s1 << 8) | (s2 << 16) | (s3 << 24);
        }
        if constexpr (WANT_MASK) out.maskbits[gi] = o.keep;
        if (out.dequant) store_dequant<T>(reinterpret_cast<T*>(out.dequant) + gi * 32, o);
    }
};

template <typename T, bool WANT_MASK>
void launch_rowmajor_g32(int mode, const void* x, int64_t rows, int64_t cols, bool tiled, float c, uint32_t sign_word,
                         uint64_t seed, const GroupOut& out, bool rotate, hipStream_t stream) {
    const T* xp = reinterpret_cast<const T*>(x);
    if (tiled) {
        const auto go = [&](auto job) { launch_job(job, stream); };
        switch (mode) {
            case QUEST_RTN: go(RowmajorTiledJob<T, QUEST_RTN, WANT_MASK>(x, rows, cols, Rotation{c, {{sign_word, 0, 0, 0}}}, seed, out)); break;
            case ABSMAX_RTN: go(RowmajorTiledJob<T, ABSMAX_RTN, WANT_MASK>(x, rows, cols, Rotation{c, {{sign_word, 0, 0, 0}}}, seed, out)); break;
            case ABSMAX_SR: go(RowmajorTiledJob<T, ABSMAX_SR, WANT_MASK>(x, rows, cols, Rotation{c, {{sign_word, 0, 0, 0}}}, seed, out)); break;
            default: go(RowmajorTiledJob<T, QUEST_SR, WANT_MASK>(x, rows, cols, Rotation{c, {{sign_word, 0, 0, 0}}}, seed, out)); break;
        }
        return;
    }
    const int64_t n_groups = rows * cols / 32;
    dim3 grid((unsigned)((n_groups + 255) / 256)), block(256);
    switch (mode) {
        case QUEST_RTN: quantize_rowmajor_g32_kernel<T, QUEST_RTN, WANT_MASK><<<grid, block, 0, stream>>>(xp, n_groups, c, sign_word, seed, out, (int)rotate); break;
        case ABSMAX_RTN: quantize_rowmajor_g32_kernel<T, ABSMAX_RTN, WANT_MASK><<<grid, block, 0, stream>>>(xp, n_groups, c, sign_word, seed, out, (int)rotate); break;
        case ABSMAX_SR: quantize_rowmajor_g32_kernel<T, ABSMAX_SR, WANT_MASK><<<grid, block, 0, stream>>>(xp, n_groups, c, sign_word, seed, out, (int)rotate); break;
        default: quantize_rowmajor_g32_kernel<T, QUEST_SR, WANT_MASK><<<grid, block, 0, stream>>>(xp, n_groups, c, sign_word, seed, out, (int)rotate); break;
    }
}

template <typename T, int MODE, bool WANT_MASK, int HD>
__global__ __launch_bounds__(256) void quantize_rowmajor_wide_kernel(const T* __restrict__ x, int64_t n_groups, float c,
                                                                     SignBits sf, uint64_t seed, GroupOut out) {
    static_assert(HD == 64 || HD == 128, "lane pairs or quads");
    job_starts();
    const int64_t gi = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gi >= n_groups) return;  // n_groups is a multiple of HD/32: the lanes of a chunk leave together
    float v[32];
    load_group<T>(x + gi * 32, v);
    job_requests_issued();
    rotate_block<HD>(v, Rotation{c, sf});
    GroupCodes o;
    quantize_group_regs<MODE, WANT_MASK>(v, seed, gi, o);
    job_stores_next();
    out.codes[gi] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
    out.scales[gi] = (uint8_t)o.scale_byte;
    if constexpr (WANT_MASK) out.maskbits[gi] = o.keep;
    if (out.dequant) store_dequant<T>(reinterpret_cast<T*>(out.dequant) + gi * 32, o);
}

template <typename T, bool WANT_MASK, int HD>
void launch_rowmajor_wide(int mode, const void* x, int64_t n, float c, const SignBits& sb, uint64_t seed,
                          const GroupOut& out, hipStream_t stream) {
    const T* xp = reinterpret_cast<const T*>(x);
    const int64_t n_groups = n / 32;
    const SignBits sf = wide_sign_fields<HD>(sb);
    dim3 grid((unsigned)((n_groups + 255) / 256)), block(256);
    switch (mode) {
        case QUEST_RTN: quantize_rowmajor_wide_kernel<T, QUEST_RTN, WANT_MASK, HD><<<grid, block, 0, stream>>>(xp, n_groups, c, sf, seed, out); break;
        case ABSMAX_RTN: quantize_rowmajor_wide_kernel<T, ABSMAX_RTN, WANT_MASK, HD><<<grid, block, 0, stream>>>(xp, n_groups, c, sf, seed, out); break;
        case ABSMAX_SR: quantize_rowmajor_wide_kernel<T, ABSMAX_SR, WANT_MASK, HD><<<grid, block, 0, stream>>>(xp, n_groups, c, sf, seed, out); break;
        default: quantize_rowmajor_wide_kernel<T, QUEST_SR, WANT_MASK, HD><<<grid, block, 0, stream>>>(xp, n_groups, c, sf, seed, out); break;
    }
}

// ---- only the values: what the quantizer modules return -------------------------------------------------------------
// One group per lane, flat over the tensor, no codes and scales written.  A wave's 64 groups are contiguous, and pass through LDS both
// ways: an instruction then moves a contiguous KiB, where a lane's own group is four (fp32: eight) 16-byte pieces 64 (128) bytes
// from its neighbour's.  Slot kPieces l + (q ^ swizzle) holds piece q of lane l's group: slot-ordered and group-ordered accesses both
// spread over all banks.  The last wave of a tensor, if it is not whole, takes its groups lane by lane.
// What bounds it: HBM.  16384 x 4096 bf16 with mask, blocks of 64: 75 us with codes and scales, every value taken apart by hand; 62
// without the former and by hardware converts; 48 with whole lines.
// past_in, past_out: loads and stores past the caches, by size: the values are what the next launch reads.  us in bf16 with a product
// by 1024 columns behind it, an elementwise reader, and the straight-through backward alone, which leaves the values unread;
// neither, loads, both:
//   8192 x 4096 (64 MiB)    77.2 79.2 84.5    42.3 43.2 46.6    60 58 60
//   16384 x 4096 (128 MiB) 129.3 130.3 137.2   84.0 82.0 86.7    101.5 87.9 90.3
//   24576 x 4096 (192 MiB) 220.9 212.0 220.9    140.4 126.3 136.5    149.6 135.2 130.4
//   32768 x 4096 (256 MiB) 267.3 261.7 268.0   184.8 186.5 183.4    197.3 177.4 174.3
//   32768 x 8192 (512 MiB) 537.7 534.3 518.4   365.8 370.0 357.8    380.0 360.6 354.0
// WANT_MASK: maskbits or null; the quest modes always work it out, as the quantizer modules want it, the absmax modes where it is asked for
template <typename T, int MODE, bool WANT_MASK, int HD>
__global__ __launch_bounds__(256) void quantize_values_kernel(const T* __restrict__ x, int64_t n_groups, Rotation rot, uint64_t seed,
                                                              uint32_t* __restrict__ maskbits, T* __restrict__ values, bool past_in, bool past_out) {
    constexpr int kPieces = 2 * (int)sizeof(T);   // 16-byte pieces per group
    job_starts();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t first = (int64_t)blockIdx.x * 256 + wave * 64, gi = first + lane;
    const bool whole = first + 64 <= n_groups;   // uniform
    if (gi >= n_groups) return;  // n_groups is a multiple of HD/32: the lanes of a chunk leave together
    uint4* area = job_lds + wave * 64 * kPieces;
    const auto swizzle = [](int l) { return sizeof(T) == 2 ? (l >> 2) & 3 : l & 7; };
    // slot 64 i + lane: piece lane % kPieces, swizzled, of group 64 i / kPieces + lane / kPieces
    const auto piece_of_slot = [&](int i) {
        const int group = (64 * i + lane) / kPieces;
        return group * kPieces + ((lane % kPieces) ^ swizzle(group));
    };
    float v[32];
    if (whole) {
        const uint4* src = reinterpret_cast<const uint4*>(x + first * 32);
        uint4 raw[kPieces];
        if (past_in) {
#pragma unroll
            for (int i = 0; i < kPieces; ++i) raw[i] = stream_load(src + piece_of_slot(i));
        } else {
#pragma unroll
            for (int i = 0; i < kPieces; ++i) raw[i] = src[piece_of_slot(i)];
        }
        job_requests_issued();
#pragma unroll
        for (int i = 0; i < kPieces; ++i) area[64 * i + lane] = raw[i];
        wave_settle();
#pragma unroll
        for (int q = 0; q < kPieces; ++q) {
            const uint4 t = area[kPieces * lane + (q ^ swizzle(lane))];
            const uint32_t w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (sizeof(T) == 2) {
                    v[q * 8 + 2 * i] = u2f(w[i] << 16);
                    v[q * 8 + 2 * i + 1] = u2f(w[i] & 0xffff0000u);
                } else {
                    v[q * 4 + i] = u2f(w[i]);
                }
            }
        }
    } else {
        load_group<T>(x + gi * 32, v);
    }
    rotate_block<HD>(v, rot);
    GroupCodes o;
    quantize_group_regs<MODE, WANT_MASK>(v, seed, gi, o);
    uint4 out[kPieces];
    group_values<T>(o, out);
    job_stores_next();
    if (WANT_MASK && maskbits) maskbits[gi] = o.keep;
    if (whole) {
        wave_settle();
#pragma unroll
        for (int q = 0; q < kPieces; ++q) area[kPieces * lane + (q ^ swizzle(lane))] = out[q];
        wave_settle();
        uint4* dst = reinterpret_cast<uint4*>(values + first * 32);
        if (past_out) {
#pragma unroll
            for (int i = 0; i < kPieces; ++i) stream_store(dst + piece_of_slot(i), area[64 * i + lane]);
        } else {
#pragma unroll
            for (int i = 0; i < kPieces; ++i) dst[piece_of_slot(i)] = area[64 * i + lane];
        }
    } else {
#pragma unroll
        for (int q = 0; q < kPieces; ++q) reinterpret_cast<uint4*>(values + gi * 32)[q] = out[q];
    }
}

// ---- transposed input: x is [P, Q] row-major, output is the [Q, P] tensor quantized along P ----------
// A workgroup owns a strip of 256 bytes of columns (128 bf16 / 64 fp32) by 128 rows; wave w owns p-group w.
// A lane reads its column (bf16: two adjacent columns per 32-bit load) at 32 successive rows straight from
// global memory: each wave load is one contiguous 256-byte row segment, 8 KiB in flight per wave, no LDS and
// no barrier on the input side.  Codes and scales go through LDS so that each q row leaves the workgroup as
// one contiguous 64-byte (codes) / 4-byte (scales) piece.
template <typename T>
struct TrTile {
    static constexpr int kQ = 256 / (int)sizeof(T);      // 128 columns of bf16, 64 of fp32
    static constexpr int kGroupsPerLane = kQ / 64;       // 2 for bf16, 1 for fp32
};
constexpr int kTrP = 128;

// Hadamard blocks 64 and 128 span two or four p-groups of a column.  Those groups then sit in neighbouring lanes (the lane
// pair or quad of rotate_block) instead of in different waves: a wave covers fewer columns and all p-groups of the block.
// PADDED: tiled codes of a P that is not a multiple of 128, completed with zero codes and scales.
template <typename T, int MODE, bool DENSE = false, int HD = 32, bool PADDED = false>
struct TransposedJob {
    static constexpr int kLds = TrTile<T>::kQ * (4 * 16 + 4);
    static constexpr int kWaves = 0;
    const T* x;
    int64_t P, Q;
    Rotation rot;
    uint64_t seed;
    const uint64_t* seed_base = nullptr;  // device memory, or null: a value the kernel adds to `seed` when it runs
    uint8_t* codes;
    uint8_t* scales;
    void* dequant;
    bool tiled_out;
    const float* matrix;  // DENSE: the rotation, [32][32] fp32 (rot is then unused)
    unsigned grid_p, blocks;

    TransposedJob(const void* x_, int64_t P_, int64_t Q_, const Rotation& rot_, uint64_t seed_, uint8_t* codes_, uint8_t* scales_,
                  void* dequant_, bool tiled_out_, const float* matrix_ = nullptr)
        : x(reinterpret_cast<const T*>(x_)), P(P_), Q(Q_), rot(rot_), seed(seed_), codes(codes_),
          scales(scales_), dequant(dequant_), tiled_out(tiled_out_), matrix(matrix_), grid_p((unsigned)((P_ + kTrP - 1) / kTrP)),
          blocks((unsigned)(((P_ + kTrP - 1) / kTrP) * ((Q_ + TrTile<T>::kQ - 1) / TrTile<T>::kQ))) {}

    __device__ __forceinline__ void run(unsigned bid) const {
        constexpr int TQ = TrTile<T>::kQ;
        constexpr int GPL = TrTile<T>::kGroupsPerLane;
        uint4* ocodes = job_lds;                                               // [q][4 groups x 16 B]
        uint8_t* oscales = reinterpret_cast<uint8_t*>(job_lds + TQ * 4);       // [q][4 B]
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // tells the compiler it is wave-uniform
        const unsigned bq = bid / grid_p;
        const int64_t p0 = (int64_t)(bid - bq * grid_p) * kTrP, q0 = (int64_t)bq * TQ;
        // this lane's p-group within the strip's four and its load column (GPL adjacent columns)
        const int pg = HD == 32 ? wave : HD == 64 ? (wave >> 1) * 2 + (lane & 1) : (lane & 3);
        const int cd = HD == 32 ? lane : HD == 64 ? (wave & 1) * 32 + (lane >> 1) : wave * 16 + (lane >> 2);
        const int64_t pbase = p0 + pg * 32;
        const int64_t qa = q0 + cd * GPL;           // this lane's first column
        const bool active = pbase < P && qa < Q;    // P % HD == 0 and Q % 8 == 0: all of a lane's (and of a chunk's) groups or none
        float v[GPL][32];
        if (active) {
            // uniform row pointers (scalar unit) + the lane's 32-bit dword offset: no per-lane 64-bit address math
            const int64_t row_dw = Q * (int64_t)sizeof(T) / 4;
            const uint32_t* row = reinterpret_cast<const uint32_t*>(x + (HD == 32 ? pbase : p0) * Q + q0);
            const uint32_t off = HD == 32 ? (uint32_t)lane : (uint32_t)(pg * 32 * row_dw + cd);
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const uint32_t w = (row + i * row_dw)[off];
                if constexpr (sizeof(T) == 2) {
                    v[0][i] = u2f(w << 16);
                    v[1][i] = u2f(w & 0xffff0000u);
                } else {
                    v[0][i] = u2f(w);
                }
            }
        } else if constexpr (DENSE) {
#pragma unroll
            for (int gq = 0; gq < GPL; ++gq)
#pragma unroll
                for (int i = 0; i < 32; ++i) v[gq][i] = 0.0f;
        }
        job_requests_issued();
        if constexpr (DENSE) {  // the matrix instruction needs the whole wave, lanes outside the tensor included
            DenseFrag frag;
            load_dense_frag(matrix, sizeof(T) == 2 ? BF16 : F32, frag);
#pragma unroll
            for (int gq = 0; gq < GPL; ++gq) dense_rotate(v[gq], frag);
        }
        if (active) {
#pragma unroll
            for (int gq = 0; gq < GPL; ++gq) {
                const int64_t gi = (qa + gq) * (P / 32) + pbase / 32;
                GroupCodes res;
                if constexpr (!DENSE) rotate_block<HD>(v[gq], rot);
                quantize_group_regs<MODE, false>(v[gq], seed_base ? seed + *seed_base : seed, gi, res);
                if (dequant) store_dequant<T>(reinterpret_cast<T*>(dequant) + gi * 32, res);
                ocodes[(cd * GPL + gq) * 4 + pg] = make_uint4(res.w[0], res.w[1], res.w[2], res.w[3]);
                oscales[(cd * GPL + gq) * 4 + pg] = (uint8_t)res.scale_byte;
            }
        } else if constexpr (PADDED) {
#pragma unroll
            for (int gq = 0; gq < GPL; ++gq) {
                ocodes[(cd * GPL + gq) * 4 + pg] = make_uint4(0u, 0u, 0u, 0u);
                oscales[(cd * GPL + gq) * 4 + pg] = 0;
            }
        }
        __syncthreads();
        const int64_t code_pitch = P / 2, P_p = PADDED ? padded_cols(P) : P, scale_pitch = P_p / 32;
        for (int idx = tid; idx < TQ * 4; idx += 256) {
            const int ql = idx >> 2, part = idx & 3;
            if (q0 + ql < Q && p0 + part * 32 < P_p) {
                // tiled: this workgroup's 128 p are one 64-byte column block, so 16 consecutive q rows form one 1 KiB tile
                const int64_t off = tiled_out ? tiled_code_offset(q0 + ql, p0 / 128, P_p / 128) + part * 16
                                              : (q0 + ql) * code_pitch + p0 / 2 + part * 16;
                *reinterpret_cast<uint4*>(codes + off) = ocodes[idx];
            }
        }
        if (tid < TQ && q0 + tid < Q) {
            const uint32_t sw = reinterpret_cast<const uint32_t*>(oscales)[tid];
            uint8_t* dst = scales + (q0 + tid) * scale_pitch + p0 / 32;
            if (p0 + kTrP <= P_p) {
                *reinterpret_cast<uint32_t*>(dst) = sw;
            } else {
                for (int b = 0; b < 4; ++b)
                    if (p0 + b * 32 < P) dst[b] = (uint8_t)(sw >> (8 * b));
            }
        }
    }
};

// ---- packed MXFP4 in, transposed + rotated + re-quantized out --------------------------------------------
// in: codes [R, C/2], scales [R, C/32]; out: the [C, R] tensor quantized along R.  A wave owns 128 rows by 64
// columns: lane l reads, for the 32 rows of row group l / 16, the two code bytes (four columns c) at byte column
// 2 (l % 16) straight from global memory -- a wave load is four contiguous 32-byte row segments, two rows share a
// register -- plus the rows' E8M0 byte of its column group.  It then handles its four columns two at a time: the
// hardware FP4 de-quantizing convert turns one byte of each row into two floats, which gives two groups of 32 along r
// in registers.  A workgroup stacks its four waves along r (512 rows), so that a column's scale bytes leave as one
// 16-byte piece; codes leave through LDS as whole 64-byte row pieces (tiled output: four contiguous 1 KiB tiles per wave).
constexpr int kRqR = 512, kRqC = 64;

// (Row-major operands, dense rotations, absmax-coded and de-quantized tensors; a layer's backward pass runs RequantTiledJob.)
template <int VAL_DTYPE, int MODE, bool DENSE = false>
struct RequantJob {
    static constexpr int kLds = 4 * kRqC * 4 * 16 + kRqC * 16;
    static constexpr int kWaves = DENSE ? 1 : 3;   // three waves on a SIMD: at 173 registers (two waves) 28 us where three take 24
    const uint8_t* codes_in;
    const uint8_t* scales_in;
    int64_t R, C;
    float post;
    Rotation rot;
    uint64_t seed;
    uint8_t* codes;
    uint8_t* scales;
    void* dequant;
    bool tiled_in, tiled_out;
    const float* matrix;  // DENSE: the rotation, [32][32] fp32 (rot is then unused)
    unsigned grid_r, blocks;

    RequantJob(const uint8_t* codes_in_, const uint8_t* scales_in_, int64_t R_, int64_t C_, float post_, const Rotation& rot_,
               uint64_t seed_, uint8_t* codes_, uint8_t* scales_, void* dequant_, bool tiled_in_, bool tiled_out_,
               const float* matrix_ = nullptr)
        : codes_in(codes_in_), scales_in(scales_in_), R(R_), C(C_), post(post_), rot(rot_), seed(seed_),
          codes(codes_), scales(scales_), dequant(dequant_), tiled_in(tiled_in_), tiled_out(tiled_out_), matrix(matrix_),
          grid_r((unsigned)((R_ + kRqR - 1) / kRqR)),
          blocks((unsigned)(((R_ + kRqR - 1) / kRqR) * ((C_ + kRqC - 1) / kRqC))) {}

    // columns 2 P and 2 P + 1 of the lane's four: de-quantize byte P of the 32 rows, rotate, quantize, stage
    template <int P>
    __device__ __forceinline__ void column_pair(const uint32_t (&cw)[16], const float (&sc)[32], const DenseFrag& frag, bool active,
                                                int64_t ca, int64_t rbase, int cq, int rg, int wave, uint4* ocodes,
                                                uint8_t* oscales) const {
        using T = typename std::conditional<VAL_DTYPE == BF16, uint16_t, float>::type;
        float v[2][32];
#pragma unroll
        for (int i = 0; i < 32; i += 2) {
            // cw[i / 2]: bytes 0, 1 = row i, bytes 2, 3 = row i + 1
            const v2f pr0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw[i >> 1], sc[i], P);
            const v2f pr1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw[i >> 1], sc[i + 1], 2 + P);
            v[0][i] = pr0.x; v[1][i] = pr0.y;
            v[0][i + 1] = pr1.x; v[1][i + 1] = pr1.y;
        }
        if (post != 1.0f) {  // absmax-coded input: value = code * 2^k * post, held in val_dtype
#pragma unroll
            for (int gq = 0; gq < 2; ++gq)
#pragma unroll
                for (int i = 0; i < 32; ++i) {
                    float a = v[gq][i] * post;
                    if constexpr (VAL_DTYPE == BF16) a = bf16_to_f32(f32_to_bf16(a));
                    v[gq][i] = a;
                }
        }
        if constexpr (DENSE) {  // the matrix instruction needs the whole wave, lanes outside the tensor included
            dense_rotate(v[0], frag);
            dense_rotate(v[1], frag);
        }
        if (!active) return;
#pragma unroll
        for (int gq = 0; gq < 2; ++gq) {
            const int64_t gi = (ca + 2 * P + gq) * (R / 32) + rbase / 32;
            GroupCodes res;
            if constexpr (!DENSE) rotate_block<32>(v[gq], rot);
            quantize_group_regs<MODE, false>(v[gq], seed, gi, res);
            if (dequant) store_dequant<T>(reinterpret_cast<T*>(dequant) + gi * 32, res);
            const int cl = 4 * cq + 2 * P + gq;
            ocodes[cl * 4 + rg] = make_uint4(res.w[0], res.w[1], res.w[2], res.w[3]);
            oscales[cl * 16 + wave * 4 + rg] = (uint8_t)res.scale_byte;
        }
    }

    __device__ __forceinline__ void run(unsigned bid) const {
        uint4* ocodes_all = job_lds;                        // per wave: [c][4 row groups x 16 B]
        uint4* oscales_all = job_lds + 4 * kRqC * 4;        // [c][16 scale bytes: wave-major, then row group]
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // tells the compiler it is wave-uniform
        const unsigned bc = bid / grid_r;
        const int64_t r0 = (int64_t)(bid - bc * grid_r) * kRqR, c0 = (int64_t)bc * kRqC;
        const int64_t in_code_pitch = C / 2, in_scale_pitch = C / 32;
        const int64_t rw = r0 + wave * 128;          // this wave's first row
        const int rg = lane >> 4, cq = lane & 15;   // row group within the wave, column quad
        const int64_t rbase = rw + 32 * rg;
        const int64_t ca = c0 + 4 * cq;              // this lane's first column
        const bool active = rbase < R && ca < C;     // R % 32 == 0 and C % 32 == 0: all of a lane's groups or none
        uint32_t cw[16];
        float sc[32];
        if (active) {
            // Uniform row pointers (scalar unit) + the lane's 32-bit byte offset: no per-lane 64-bit address math.
            // Tiled input: rows are 64 bytes apart inside a 16-row block, blocks (C / 128) KiB apart.
            const int64_t blk = (C / 128) * 1024;
            const uint8_t* cu = tiled_in ? codes_in + tiled_code_offset(rw, c0 / 128, C / 128) + (c0 & 127) / 2
                                         : codes_in + rw * in_code_pitch + c0 / 2;
            const uint32_t lane_off = (uint32_t)((tiled_in ? 2 * rg * blk : 32 * rg * in_code_pitch) + 2 * cq);
            const int64_t row_step = tiled_in ? 64 : in_code_pitch;                 // next row of a 16-row block
            const int64_t block_step = tiled_in ? blk - 16 * 64 : 0;                // extra hop into the next block
            const uint8_t* su = scales_in + rw * in_scale_pitch + c0 / 32;
            const uint32_t slane_off = (uint32_t)(32 * rg * in_scale_pitch + (cq >> 3));
#pragma unroll
            for (int i = 0; i < 32; i += 2) {
                const uint32_t lo = *reinterpret_cast<const uint16_t*>(cu + i * row_step + (i >> 4) * block_step + lane_off);
                const uint32_t hi = *reinterpret_cast<const uint16_t*>(cu + (i + 1) * row_step + (i >> 4) * block_step + lane_off);
                cw[i >> 1] = lo | (hi << 16);
            }
#pragma unroll
            for (int i = 0; i < 32; ++i) sc[i] = u2f((uint32_t)(su + i * in_scale_pitch)[slane_off] << 23);
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) cw[i] = 0u;
#pragma unroll
            for (int i = 0; i < 32; ++i) sc[i] = 1.0f;
        }
        job_requests_issued();
        DenseFrag frag;
        if constexpr (DENSE) load_dense_frag(matrix, VAL_DTYPE, frag);
        uint4* ocodes = ocodes_all + wave * (kRqC * 4);
        uint8_t* oscales = reinterpret_cast<uint8_t*>(oscales_all);
        column_pair<0>(cw, sc, frag, active, ca, rbase, cq, rg, wave, ocodes, oscales);
        column_pair<1>(cw, sc, frag, active, ca, rbase, cq, rg, wave, ocodes, oscales);
        __syncthreads();
        const int64_t code_pitch = R / 2, scale_pitch = R / 32;
        // codes: each wave writes its own 64 x 64-byte tile
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int idx = it * 64 + lane, cl = idx >> 2, part = idx & 3;
            if (c0 + cl < C && rw + part * 32 < R) {
                const int64_t off = tiled_out ? tiled_code_offset(c0 + cl, rw / 128, R / 128) + part * 16
                                              : (c0 + cl) * code_pitch + rw / 2 + part * 16;
                *reinterpret_cast<uint4*>(codes + off) = ocodes[idx];
            }
        }
        // scales: one column's 16 bytes (the workgroup's 512 rows) per thread
        if (tid < kRqC && c0 + tid < C) {
            const uint4 sw = oscales_all[tid];
            uint8_t* dst = scales + (c0 + tid) * scale_pitch + r0 / 32;
            if (r0 + kRqR <= R && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
                *reinterpret_cast<uint4*>(dst) = sw;
            } else {
                const uint32_t w4[4] = {sw.x, sw.y, sw.z, sw.w};
                for (int b = 0; b < 16; ++b)
                    if (r0 + b * 32 < R) dst[b] = (uint8_t)(w4[b >> 2] >> (8 * (b & 3)));
            }
        }
    }
};

// ---- the same for a layer's backward pass: tiled quest-coded operands, rotated on the matrix pipe -----------------------
// One wave owns 128 rows by 64 columns, a workgroup four of them stacked along r, as above.  A wave requests its codes global ->
// LDS (16-byte pieces) and a scale byte pair per row; the transposing LDS read for 4-bit data hands lane l the 32 codes of column
// l, k-contiguous, which is how the scaled matrix instruction reads its FP4 operand.  The other operand is the Hadamard matrix
// with the rows' scales on it: A[j][k] = +-2^(E_k), an eight-bit E5M2 value whose exponent field is the scale byte less a base.
// So 32 rows x 32 columns are de-quantized, transposed and rotated by one instruction (K = 32 of its 64: columns 32..63 use the
// other half of A), and two results and sixteen lane-half swaps give every lane the rotated group of its column.
// Exact: the sums are multiples of half the smallest scale, and while the block's scales span at most ten octaves the instruction
// adds them without a rounding (2 M random sums of K = 32 and 64 compared with exact ones: none differs up to 10, half of them
// at 12), so that any order of additions, the butterfly's among them, gives the same fp32 values.  A block with more spread
// (or scales near the ends of the range) takes rotate_block, its groups in neighbouring lanes, and stores its codes by itself: a row of
// zeros (scale 2^-27) among others sends its Hadamard block of rows there.  Steps with 5 % of the tokens zero, in us (none zero; on the
// kernel above, either way): 16480 x 1728 x 640 131 (124; 152), 8192 x 4096 x 4096 294 (289; 298), with blocks of 64 333 (327; 338), of
// 128 337 (330; 345), 16512 x 1792 x 640 with blocks of 128 140 (133; 171).  Zero rows together, as padding behind the tokens, cost nothing.
// What bounds it: vector instructions (385 a group, 0.7 us per wave and group of 32 at 2.4 GHz, half of that Philox and the
// stochastic converts); a row group's codes are waited for when they are needed.  It runs in one grid with the quantizers of the
// error signal (backward_waves).  Both operands of a layer in a grid of their own, 8192 x 4096 and 11008 x 4096: 46 us; 16384 x 4096 and
// 1536 x 4096: 43; 16480 x 1728 and 640 x 1728: 22.  The kernel above (544 instructions a group, 64 narrow loads per lane, three waves on a
// SIMD) took 56, 53 and 26.  The four jobs of 8192 x 4096 x 4096 in one grid take 68 us, in two 71.
template <int MODE, int HD, bool PADDED>
struct RequantTiledJob {
    static constexpr int kRegion = 128 * 32;                                     // a wave's codes, in and out
    static constexpr int kScalesIn = 4 * kRegion, kScalesOut = kScalesIn + 4 * 256;
    static constexpr int kLds = kScalesOut + kRqC * 16;
    static constexpr int kWaves = backward_waves(HD);
    static constexpr int P = HD / 32;                                            // groups of a Hadamard block
    const uint8_t* codes_in;
    const uint8_t* scales_in;
    int64_t R, C;
    SignBits signs;
    Rotation rot;         // of rotate_block
    uint64_t seed;
    const uint64_t* seed_base;   // device memory, or null: a value the kernel adds to `seed` when it runs
    uint8_t* codes;
    uint8_t* scales;
    unsigned grid_r, blocks;

    RequantTiledJob(const RequantArgs& a, const SignBits& signs_, const uint64_t* seed_base_)
        : codes_in(a.codes_in), scales_in(a.scales_in), R(a.R), C(a.C), signs(signs_), rot(make_rotation<HD>(a.val_dtype, signs_)),
          seed(a.seed), seed_base(seed_base_), codes(a.codes), scales(a.scales), grid_r((unsigned)((a.R + kRqR - 1) / kRqR)),
          blocks((unsigned)(((a.R + kRqR - 1) / kRqR) * ((a.C + kRqC - 1) / kRqC))) {}

    typedef int v2i __attribute__((ext_vector_type(2)));
    typedef int v8i __attribute__((ext_vector_type(8)));
    typedef uint16_t v2u16 __attribute__((ext_vector_type(2)));

    // largest value of either half over the lanes of a half-wave, in every lane of it
    __device__ __forceinline__ static v2u16 half_wave_max(v2u16 x) {
        const auto with = [](v2u16 v, int other) { return __builtin_elementwise_max(v, __builtin_bit_cast(v2u16, other)); };
        x = with(x, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, true));    // quad_perm [1,0,3,2]
        x = with(x, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x4E, 0xf, 0xf, true));    // quad_perm [2,3,0,1]
        x = with(x, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x141, 0xf, 0xf, true));   // row_half_mirror
        x = with(x, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x140, 0xf, 0xf, true));   // row_mirror
        const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x), false, false);
        return with(__builtin_bit_cast(v2u16, r[0]), (int)r[1]);
    }

    // a block of scales with too wide a spread: groups chunk * P .. + P - 1 of the wave's 64 columns
    __device__ __forceinline__ void wide_spread(int chunk, const uint8_t* region, const uint8_t* scales_lds, uint8_t* scales_out, int lane,
                                                int64_t rw, int64_t c0, int64_t R_p, uint64_t s) const {
        const int g = chunk * P + (lane & (P - 1));
#pragma unroll 1
        for (int pass = 0; pass < P; ++pass) {
            const int col = pass * (64 / P) + lane / P;
            // the group's codes and scale bytes, packed: few registers, for a path that is rarely taken
            uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < 32; ++i) w[i >> 3] |= ((uint32_t)region[(32 * g + i) * 32 + col / 2] >> (4 * (col & 1)) & 15u) << (4 * (i & 7));
            const uint4* e = reinterpret_cast<const uint4*>(scales_lds + (col >> 5) * 128 + 32 * g);
            const uint4 e0 = e[0], e1 = e[1];
            const uint32_t sc[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
            float v[32];
#define QM_DEQUANT(I)                                                                                                              \
    v[I] = v2f(__builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[(I) >> 3], u2f((sc[(I) >> 2] >> (8 * ((I) & 3)) & 0xffu) << 23), ((I) >> 1) & 3)).x;       \
    v[(I) + 1] = v2f(__builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[(I) >> 3], u2f((sc[(I) >> 2] >> (8 * (((I) + 1) & 3)) & 0xffu) << 23), ((I) >> 1) & 3)).y;
            QM_DEQUANT(0) QM_DEQUANT(2) QM_DEQUANT(4) QM_DEQUANT(6) QM_DEQUANT(8) QM_DEQUANT(10) QM_DEQUANT(12) QM_DEQUANT(14)
            QM_DEQUANT(16) QM_DEQUANT(18) QM_DEQUANT(20) QM_DEQUANT(22) QM_DEQUANT(24) QM_DEQUANT(26) QM_DEQUANT(28) QM_DEQUANT(30)
#undef QM_DEQUANT
            rotate_block<HD>(v, rot);
            GroupCodes res;
            quantize_group_regs<MODE, false>(v, s, (c0 + col) * (R / 32) + rw / 32 + g, res);
            if (c0 + col < C)
                *reinterpret_cast<uint4*>(codes + tiled_code_offset(c0 + col, rw / 128, R_p / 128) + g * 16) = make_uint4(res.w[0], res.w[1], res.w[2], res.w[3]);
            scales_out[col * 16 + g] = (uint8_t)res.scale_byte;
        }
    }

    __device__ __forceinline__ void run(unsigned bid) const {
        uint8_t* lds = reinterpret_cast<uint8_t*>(job_lds);
        const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint4*)job_lds;
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // tells the compiler it is wave-uniform
        const unsigned bc = bid / grid_r;
        const int64_t r0 = (int64_t)(bid - bc * grid_r) * kRqR, c0 = (int64_t)bc * kRqC;
        const int64_t C_p = PADDED ? padded_cols(C) : C, R_p = PADDED ? padded_cols(R) : R;
        const int64_t rw = r0 + wave * 128;          // this wave's first row
        uint8_t* region = lds + wave * kRegion;
        uint8_t* scales_lds = lds + kScalesIn + wave * 256;              // [2 column groups][128 rows]
        uint8_t* scales_out = lds + kScalesOut + wave * 4;               // [64 columns][16]: this wave's four bytes
        if (rw < R) {
            const int rows = (int)(R - rw < 128 ? R - rw : 128);         // a multiple of 32
            const uint32_t scale_pitch_in = (uint32_t)(C_p / 32);
            const uint8_t* su = scales_in + rw * scale_pitch_in + c0 / 32;
            const auto row_of = [&](int r) { return (uint32_t)(!PADDED || r < rows ? r : rows - 1) * scale_pitch_in; };
            const uint32_t blk = (uint32_t)(C_p / 128) * 1024u;
            const uint8_t* cu = codes_in + tiled_code_offset(rw, c0 / 128, C_p / 128) + (c0 & 127) / 2;
            const int last = PADDED ? (int)((padded_rows(R) - rw) / 16) - 1 : 7;
            const auto rows_at = [&](int i) {   // request i: row group i, a row's 32 bytes in two neighbouring lanes
                const int b = 2 * i + (lane >> 5);
                return (uint32_t)(PADDED && b > last ? last : b) * blk + (uint32_t)(((lane >> 1) & 15) * 64 + (lane & 1) * 16);
            };
            const uint32_t to = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_base + wave * kRegion));
            // the scale byte pairs of rows lane and 64 + lane (both column groups), then the codes.  One statement, which ends when
            // the scales are in: left to the compiler, waiting for them would be waiting for everything.
            uint32_t sa, sb;
            asm volatile("global_load_ushort %0, %2, %4\n\tglobal_load_ushort %1, %3, %4\n\t"
                         "s_mov_b32 m0, %9\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %13\n\t"
                         "s_mov_b32 m0, %10\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %6, %13\n\t"
                         "s_mov_b32 m0, %11\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %7, %13\n\t"
                         "s_mov_b32 m0, %12\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %8, %13\n\t"
                         "s_setprio 0\n\ts_waitcnt vmcnt(4)"
                         : "=&v"(sa), "=&v"(sb)
                         : "v"(row_of(lane)), "v"(row_of(64 + lane)), "s"(su), "v"(rows_at(0)), "v"(rows_at(1)), "v"(rows_at(2)), "v"(rows_at(3)), "s"(to),
                           "s"(to + 1024u), "s"(to + 2048u), "s"(to + 3072u), "s"(cu)
                         : "memory");
            if (PADDED && c0 + 32 >= C) {   // C % 64 == 32: the second column group is padding
                sa = (sa & 0xffu) * 0x101u;
                sb = (sb & 0xffu) * 0x101u;
            }
            const uint64_t s = seed_base ? seed + *seed_base : seed;
            scales_lds[lane] = (uint8_t)sa;
            scales_lds[128 + lane] = (uint8_t)(sa >> 8);
            scales_lds[64 + lane] = (uint8_t)sb;
            scales_lds[192 + lane] = (uint8_t)(sb >> 8);
            // extremes of the scales of each row group and column group (low half: columns 0..31)
            const auto halves = [](uint32_t b) { return __builtin_bit_cast(v2u16, (b & 0xffu) | (b & 0xff00u) << 8); };
            const v2u16 full = {255, 255};
            const v2u16 hi_a = half_wave_max(halves(sa)), hi_b = half_wave_max(halves(sb));
            const v2u16 lo_a = half_wave_max(full - halves(sa)), lo_b = half_wave_max(full - halves(sb));
            uint32_t smin[2] = {0u, 0u};   // per column group: byte c = smallest scale of chunk c (the row groups of a Hadamard block)
            uint32_t fast = 0u;            // chunks whose scales are close enough together
#pragma unroll
            for (int c = 0; c < 4 / P; ++c) {
                bool ok = true;
#pragma unroll
                for (int cg = 0; cg < 2; ++cg) {
                    uint32_t top = 0u, bottom = 0u;   // largest scale, largest 255 - scale
#pragma unroll
                    for (int g = c * P; g < c * P + P; ++g) {
                        const uint32_t h = (uint32_t)__builtin_amdgcn_readlane(__builtin_bit_cast(int, g < 2 ? hi_a : hi_b), 32 * (g & 1)) >> (16 * cg) & 0xffu;
                        const uint32_t l = (uint32_t)__builtin_amdgcn_readlane(__builtin_bit_cast(int, g < 2 ? lo_a : lo_b), 32 * (g & 1)) >> (16 * cg) & 0xffu;
                        top = h > top ? h : top;
                        bottom = l > bottom ? l : bottom;
                    }
                    const uint32_t low = 255u - bottom;
                    smin[cg] |= low << (8 * c);
                    ok = ok && top - low <= 10u && low >= 32u && top <= 240u;
                }
                fast |= (ok ? 1u : 0u) << c;
            }
            wave_settle();
            // results: piece g of column l at slot l ^ 2 g of the KiB that held row group g's codes
            uint4* stage = reinterpret_cast<uint4*>(region);
            const auto rotate_chunk = [&](int c, int lane) {
                // the signs of A's bytes: lane (j, half h) holds S[j][16 h + 4 d + q] in byte q of dword d
                uint32_t hs[4];
                {
                    const uint32_t j = (uint32_t)lane;
                    const uint32_t all = 0x80808080u;
                    const uint32_t quad = (j & 1u) << 15 | (j & 2u) << 22 | ((j ^ (j >> 1)) & 1u) << 31;
                    const uint32_t t = quad ^ ((j & 16u) && (j & 32u) ? all : 0u);
                    hs[0] = t;
                    hs[1] = t ^ ((j & 4u) ? all : 0u);
                    hs[2] = t ^ ((j & 8u) ? all : 0u);
                    hs[3] = hs[1] ^ ((j & 8u) ? all : 0u);
                }
                const uint32_t low[2] = {smin[0] >> (8 * c) & 0xffu, smin[1] >> (8 * c) & 0xffu};
                v2i b[P][2];
                uint32_t ex[P][2][4];
#pragma unroll
                for (int kb = 0; kb < P; ++kb) {
                    const int g = c * P + kb;
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        b[kb][q] = __builtin_amdgcn_ds_read_tr4_b64_v2i32(
                            (__attribute__((address_space(3))) v2i*)(uintptr_t)(lds_base + wave * kRegion + (32 * g + 16 * q + (lane & 15)) * 32 + (lane >> 4) * 8));
#pragma unroll
                    for (int cg = 0; cg < 2; ++cg) {
                        const uint4 e = *reinterpret_cast<const uint4*>(scales_lds + cg * 128 + 32 * g + 16 * (lane >> 5));
                        const uint32_t w[4] = {e.x, e.y, e.z, e.w};
                        // exponent fields 1 .. 11 of E5M2 bytes: no byte carries into the next
                        const uint32_t base = (low[cg] - 1u) * 0x04040404u;
#pragma unroll
                        for (int d = 0; d < 4; ++d) ex[kb][cg][d] = (w[d] << 2) - base;
                    }
                }
#pragma unroll 1
                for (int ob = 0; ob < P; ++ob) {
                    v16f d0, d1;
#pragma unroll
                    for (int e = 0; e < 16; ++e) d0[e] = d1[e] = 0.0f;
#pragma unroll
                    for (int kb = 0; kb < P; ++kb) {
                        const uint32_t flip = (__builtin_popcount((unsigned)(ob & kb)) & 1) ? 0x80808080u : 0u;
                        const v8i codes_k = v8i{b[kb][0].x, b[kb][0].y, b[kb][1].x, b[kb][1].y, 0, 0, 0, 0};
                        const auto a = [&](int cg, int d) { return (int)xor3(ex[kb][cg][d], hs[d], flip); };
                        // scale bytes: A's values are 2^(field - 15) = 2^(S - low - 14); codes carry none (127)
                        int z[4];   // zeros that do not hold registers from one iteration to the next
                        asm volatile("v_mov_b32 %0, 0\n\tv_mov_b32 %1, 0\n\tv_mov_b32 %2, 0\n\tv_mov_b32 %3, 0" : "=v"(z[0]), "=v"(z[1]), "=v"(z[2]), "=v"(z[3]));
                        d0 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v8i{a(0, 0), a(0, 1), a(0, 2), a(0, 3), z[0], z[1], z[2], z[3]}, codes_k, d0, 1, 4, 0,
                                                                             (int)(low[0] + 14u), 0, 127);
                        d1 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v8i{z[0], z[1], z[2], z[3], a(1, 0), a(1, 1), a(1, 2), a(1, 3)}, codes_k, d1, 1, 4, 0,
                                                                             (int)(low[1] + 14u), 0, 127);
                    }
                    // element e of a lane's result is row j = 8 (e / 4) + 4 (lane / 32) + e % 4 of column lane % 32 (+ 32 for d1)
                    float v[32];
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const auto r = __builtin_amdgcn_permlane32_swap(f2u(d0[e]), f2u(d1[e]), false, false);
                        v[8 * (e / 4) + (e % 4)] = u2f(r[0]);
                        v[8 * (e / 4) + 4 + (e % 4)] = u2f(r[1]);
                    }
                    scale_group(v, rot.c, ob == 0 ? signs.w[0] : ob == 1 ? signs.w[1] : ob == 2 ? signs.w[2] : signs.w[3]);
                    const int g = c * P + ob;
                    GroupCodes res;
                    quantize_group_regs<MODE, false>(v, s, (c0 * (R / 32) + rw / 32 + g) + (uint32_t)(lane * (int)(R / 32)), res);
                    stage[64 * g + (lane ^ (2 * g))] = make_uint4(res.w[0], res.w[1], res.w[2], res.w[3]);
                    scales_out[lane * 16 + g] = (uint8_t)res.scale_byte;
                }
            };
            uint32_t staged = 0u;   // row groups whose codes pass through LDS: all but those of wide_spread
#pragma unroll 1
            for (int c = 0; c < 4 / P; ++c) {
                // an opaque copy: what is worked out from it stays inside the loop instead of holding registers across it
                int lane = (int)threadIdx.x & 63;
                asm volatile("" : "+v"(lane));
                // row group i is the wave's i-th request of codes: this chunk's are in once at most the later groups' are pending
                // (a store may be among the pending ones: the wait is then longer, not shorter)
                if (c == 0) __builtin_amdgcn_s_waitcnt(vmcnt_imm(4 - P));
                else if (P == 1 && c == 1) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2));
                wave_settle();
                const bool inside = !PADDED || 32 * c * P < rows;   // otherwise padding: zero codes and scales
                if (inside && !(fast >> c & 1u)) {
                    wide_spread(c, region, scales_lds, scales_out, lane, rw, c0, R_p, s);
                } else if (!inside) {
                    staged |= ((1u << P) - 1u) << (c * P);
#pragma unroll
                    for (int g = c * P; g < c * P + P; ++g) {
                        stage[64 * g + (lane ^ (2 * g))] = make_uint4(0u, 0u, 0u, 0u);
                        scales_out[lane * 16 + g] = 0;
                    }
                } else {
                    staged |= ((1u << P) - 1u) << (c * P);
                    rotate_chunk(c, lane);
                }
                // two row groups' codes leave together, 32 bytes per column (all requests have been waited for by then)
                if (P > 1 || (c & 1)) {
                    if (c == (P == 1 ? 1 : 0)) __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
                    wave_settle();
#pragma unroll
                    for (int h = 0; h < (P == 4 ? 2 : 1); ++h) {
                        const int pair = P == 4 ? h : P == 2 ? c : c >> 1;
#pragma unroll
                        for (int it = 0; it < 2; ++it) {
                            const int idx = it * 64 + lane, cl = idx >> 1, g = 2 * pair + (idx & 1);
                            if (c0 + cl < C && (staged >> g & 1u))
                                *reinterpret_cast<uint4*>(codes + tiled_code_offset(c0 + cl, rw / 128, R_p / 128) + g * 16) = stage[64 * g + (cl ^ (2 * g))];
                        }
                    }
                }
            }
        }
        __syncthreads();
        // scales: one column's 16 bytes (the workgroup's 512 rows) per thread
        if (tid < kRqC && c0 + tid < C) {
            const uint4 sw = *reinterpret_cast<const uint4*>(lds + kScalesOut + tid * 16);
            uint8_t* dst = scales + (c0 + tid) * (R_p / 32) + r0 / 32;
            if (r0 + kRqR <= R && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
                *reinterpret_cast<uint4*>(dst) = sw;
            } else {   // whole dwords: the row count is padded to 128
                const uint32_t w4[4] = {sw.x, sw.y, sw.z, sw.w};
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (r0 + j * 128 < R) *reinterpret_cast<uint32_t*>(dst + 4 * j) = w4[j];
            }
        }
    }
};

template <typename T, bool DENSE>
void launch_transposed_g32(int mode, const void* x, int64_t P, int64_t Q, const Rotation& rot, uint64_t seed,
                           uint8_t* codes, uint8_t* scales, void* dequant, bool tiled, const float* matrix, hipStream_t stream) {
    switch (mode) {
        case QUEST_RTN: launch_job(TransposedJob<T, QUEST_RTN, DENSE>(x, P, Q, rot, seed, codes, scales, dequant, tiled, matrix), stream); break;
        case ABSMAX_RTN: launch_job(TransposedJob<T, ABSMAX_RTN, DENSE>(x, P, Q, rot, seed, codes, scales, dequant, tiled, matrix), stream); break;
        case ABSMAX_SR: launch_job(TransposedJob<T, ABSMAX_SR, DENSE>(x, P, Q, rot, seed, codes, scales, dequant, tiled, matrix), stream); break;
        default: launch_job(TransposedJob<T, QUEST_SR, DENSE>(x, P, Q, rot, seed, codes, scales, dequant, tiled, matrix), stream); break;
    }
}

template <int VAL_DTYPE, bool DENSE>
void launch_requant_g32(int mode, const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C, float post,
                        const Rotation& rot, uint64_t seed, uint8_t* codes, uint8_t* scales, void* dequant,
                        bool tiled_in, bool tiled_out, const float* matrix, hipStream_t stream) {
    switch (mode) {
        case QUEST_RTN: launch_job(RequantJob<VAL_DTYPE, QUEST_RTN, DENSE>(codes_in, scales_in, R, C, post, rot, seed, codes, scales, dequant, tiled_in, tiled_out, matrix), stream); break;
        case ABSMAX_RTN: launch_job(RequantJob<VAL_DTYPE, ABSMAX_RTN, DENSE>(codes_in, scales_in, R, C, post, rot, seed, codes, scales, dequant, tiled_in, tiled_out, matrix), stream); break;
        case ABSMAX_SR: launch_job(RequantJob<VAL_DTYPE, ABSMAX_SR, DENSE>(codes_in, scales_in, R, C, post, rot, seed, codes, scales, dequant, tiled_in, tiled_out, matrix), stream); break;
        default: launch_job(RequantJob<VAL_DTYPE, QUEST_SR, DENSE>(codes_in, scales_in, R, C, post, rot, seed, codes, scales, dequant, tiled_in, tiled_out, matrix), stream); break;
    }
}

}  // namespace

// hd = 32, row-major input, RTN or Philox-driven SR (explicit uniforms take the generic path); rotate = false
// quantizes groups of 32 as they are (input rotated by the caller)
hipError_t quantize_rowmajor_hd32(const void* x, int dtype, int64_t rows, int64_t cols, uint32_t sign_word, int mode,
                                  uint64_t seed, uint8_t* codes, uint8_t* scales, uint8_t* maskbits, void* dequant,
                                  bool tiled, bool rotate, hipStream_t stream) {
    if (!rotate && (tiled || sign_word)) return hipErrorInvalidValue;  // pass-through groups: row-major codes, no signs
    GroupOut out{reinterpret_cast<uint4*>(codes), scales, reinterpret_cast<uint32_t*>(maskbits), dequant};
    const float c = rotate ? hadamard_scale(32, dtype) : 1.0f;
    if (maskbits) {
        if (dtype == BF16) launch_rowmajor_g32<uint16_t, true>(mode, x, rows, cols, tiled, c, sign_word, seed, out, rotate, stream);
        else launch_rowmajor_g32<float, true>(mode, x, rows, cols, tiled, c, sign_word, seed, out, rotate, stream);
    } else {
        if (dtype == BF16) launch_rowmajor_g32<uint16_t, false>(mode, x, rows, cols, tiled, c, sign_word, seed, out, rotate, stream);
        else launch_rowmajor_g32<float, false>(mode, x, rows, cols, tiled, c, sign_word, seed, out, rotate, stream);
    }
    return hipGetLastError();
}

// hd = 64 or 128, row-major input, RTN or Philox-driven SR, row-major codes
hipError_t quantize_rowmajor_wide(const void* x, int dtype, int64_t n, int hd, const SignBits& sb, int mode, uint64_t seed,
                                  uint8_t* codes, uint8_t* scales, uint8_t* maskbits, void* dequant, hipStream_t stream) {
    GroupOut out{reinterpret_cast<uint4*>(codes), scales, reinterpret_cast<uint32_t*>(maskbits), dequant};
    const float c = hadamard_scale(hd, dtype);
    const auto go = [&](auto tag, auto mask, auto hdc) {
        using T = decltype(tag);
        launch_rowmajor_wide<T, decltype(mask)::value, decltype(hdc)::value>(mode, x, n, c, sb, seed, out, stream);
    };
    const auto by_hd = [&](auto tag, auto mask) {
        if (hd == 64) go(tag, mask, std::integral_constant<int, 64>{});
        else go(tag, mask, std::integral_constant<int, 128>{});
    };
    if (maskbits) {
        if (dtype == BF16) by_hd(uint16_t{}, std::true_type{});
        else by_hd(float{}, std::true_type{});
    } else {
        if (dtype == BF16) by_hd(uint16_t{}, std::false_type{});
        else by_hd(float{}, std::false_type{});
    }
    return hipGetLastError();
}

// hd = 32, x is [P, Q] row-major and the output is its transpose quantized along P; no clip mask
hipError_t quantize_transposed_hd32(const void* x, int dtype, int64_t P, int64_t Q, uint32_t sign_word, int mode,
                                    uint64_t seed, uint8_t* codes, uint8_t* scales, void* dequant, bool tiled,
                                    hipStream_t stream) {
    const Rotation rot{hadamard_scale(32, dtype), {{sign_word, 0, 0, 0}}};
    if (dtype == BF16) launch_transposed_g32<uint16_t, false>(mode, x, P, Q, rot, seed, codes, scales, dequant, tiled, nullptr, stream);
    else launch_transposed_g32<float, false>(mode, x, P, Q, rot, seed, codes, scales, dequant, tiled, nullptr, stream);
    return hipGetLastError();
}

hipError_t requantize_transposed_hd32(const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C, float post,
                                      int val_dtype, uint32_t sign_word, int mode, uint64_t seed, uint8_t* codes,
                                      uint8_t* scales, void* dequant, bool tiled_in, bool tiled_out, hipStream_t stream) {
    const Rotation rot{hadamard_scale(32, val_dtype), {{sign_word, 0, 0, 0}}};
    if (val_dtype == BF16) launch_requant_g32<BF16, false>(mode, codes_in, scales_in, R, C, post, rot, seed, codes, scales, dequant, tiled_in, tiled_out, nullptr, stream);
    else launch_requant_g32<F32, false>(mode, codes_in, scales_in, R, C, post, rot, seed, codes, scales, dequant, tiled_in, tiled_out, nullptr, stream);
    return hipGetLastError();
}

// ---- the same three with a dense 32x32 rotation (matrix: device pointer to [32][32] fp32, H[k][j]; its entries are
// rounded to the tensor's dtype as the reference casts its matrix, quantizers/mxfp4.py:49) ---------------------------
hipError_t quantize_rowmajor_dense(const void* x, int dtype, int64_t rows, int64_t cols, const float* matrix, int mode,
                                   uint64_t seed, uint8_t* codes, uint8_t* scales, uint8_t* maskbits, void* dequant,
                                   bool tiled, hipStream_t stream) {
    GroupOut out{reinterpret_cast<uint4*>(codes), scales, reinterpret_cast<uint32_t*>(maskbits), dequant};
    if (maskbits) {
        if (dtype == BF16) launch_rowmajor_dense<uint16_t, true>(mode, x, rows, cols, matrix, seed, out, tiled, stream);
        else launch_rowmajor_dense<float, true>(mode, x, rows, cols, matrix, seed, out, tiled, stream);
    } else {
        if (dtype == BF16) launch_rowmajor_dense<uint16_t, false>(mode, x, rows, cols, matrix, seed, out, tiled, stream);
        else launch_rowmajor_dense<float, false>(mode, x, rows, cols, matrix, seed, out, tiled, stream);
    }
    return hipGetLastError();
}

hipError_t quantize_transposed_dense(const void* x, int dtype, int64_t P, int64_t Q, const float* matrix, int mode,
                                     uint64_t seed, uint8_t* codes, uint8_t* scales, void* dequant, bool tiled,
                                     hipStream_t stream) {
    if (dtype == BF16) launch_transposed_g32<uint16_t, true>(mode, x, P, Q, Rotation{}, seed, codes, scales, dequant, tiled, matrix, stream);
    else launch_transposed_g32<float, true>(mode, x, P, Q, Rotation{}, seed, codes, scales, dequant, tiled, matrix, stream);
    return hipGetLastError();
}

hipError_t requantize_transposed_dense(const uint8_t* codes_in, const uint8_t* scales_in, int64_t R, int64_t C, float post,
                                       int val_dtype, const float* matrix, int mode, uint64_t seed, uint8_t* codes,
                                       uint8_t* scales, void* dequant, bool tiled_in, bool tiled_out, hipStream_t stream) {
    if (val_dtype == BF16) launch_requant_g32<BF16, true>(mode, codes_in, scales_in, R, C, post, Rotation{}, seed, codes, scales, dequant, tiled_in, tiled_out, matrix, stream);
    else launch_requant_g32<F32, true>(mode, codes_in, scales_in, R, C, post, Rotation{}, seed, codes, scales, dequant, tiled_in, tiled_out, matrix, stream);
    return hipGetLastError();
}

// ---- producers fused into the forward quantizer ------------------------------------------------------------------
// The tensor the model would hand to the quantized linear (RMSNorm output, src/models/llama.py:64-75; SwiGLU product,
// llama.py:113-114) is computed group by group in registers and never written.  One wave owns one row: lane l takes
// groups l, l+64, ... of 32 consecutive elements, so a row of up to 2048 elements is read exactly once.

namespace {

// TA = void: plain.  Otherwise the norm's input is x + add (the residual sum in front of the norm, src/models/llama.py:
// 170-171), formed here in T's arithmetic and written to xsum, which the rest of the model continues with.
template <typename T, typename TA = void>
struct RmsNormProducer {
    static constexpr int kOutDtype = F32;  // bf16-or-fp32 normalised value times the fp32 gain is fp32
    static constexpr bool kAdd = !std::is_void<TA>::value;
    using TAdd = typename std::conditional<kAdd, TA, T>::type;
    static constexpr bool kWithWeight = sizeof(T) == 4 && (!kAdd || sizeof(TAdd) == 2);
    static constexpr bool kStaged = sizeof(T) == 4;
    static constexpr int kLds = kStaged ? 4 * 512 * 16 : 0;
    const T* x;
    const float* gain;
    float* factor;  // [rows]: 1 / sqrt(mean(x^2) + eps), kept for the backward pass
    float eps;
    const TAdd* add;
    T* xsum;

    // 8 KiB of LDS per wave, through which fp32 rows and the gain pass on their way to the lanes that own their groups: an
    // instruction then reads or writes whole 128-byte lines, where a lane's own 128 bytes are eight 16-byte pieces, each
    // instruction touching 64 lines, which the address unit takes one by one.  Slot 8 l + (q ^ l % 8) holds piece q of lane l's
    // group: slot-ordered and group-ordered accesses both spread over all banks.  With the residual sum, inputs cycled through
    // memory: 4096 x 640 11.7 -> 9.9 us, 16384 x 1536 62 -> 57 (4.7 TB/s; 65 -> 60 inside a layer's step), 32768 x 1024 88 -> 75,
    // 16384 x 4096 166 -> 156 (two passes); 512 x 4096 is latency, 11 us either way.  Requests under per-lane predicates instead
    // of clamped ones cost half as much again.
    // 121 to 126 registers with a bf16 summand, four waves on a SIMD: the pieces' offsets are one register each, and the gain is requested
    // when the row has left its own registers (with addresses per tensor and the gain asked for at the start: 133 and 160, three waves).
    // us inside a layer's step: 32768 x 1024 75.0 -> 65.7, 20000 x 704 36.0 -> 32.2, 16384 x 1536 with the weight 62.0 -> 59.7; latency, the
    // same either way, at 2048 x 2048 14.4 and 4096 x 640 10.
    typedef float v4 __attribute__((ext_vector_type(4)));
    typedef uint32_t w2 __attribute__((ext_vector_type(2)));
    __device__ __forceinline__ static v4* area() { return reinterpret_cast<v4*>(job_lds) + (threadIdx.x >> 6) * 512; }
    __device__ __forceinline__ static void read_group(int of_lane, float (&v)[32]) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const v4 t = area()[8 * of_lane + (q ^ (of_lane & 7))];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * q + e] = t[e];
        }
    }

    // The row's factor; `first` leaves with the raw elements of the lane's first group (if it has one).
    // Sum of squares in a fixed order: sixteen interleaved partial sums (partial j adds the sums of groups j, j+16,
    // j+32, ... in ascending order, each group summed by the pairwise tree), then the pairwise tree over the sixteen.
    // A lane without a group adds +0, which leaves a sum of squares unchanged.
    // W < 64: the wave holds 64 / W rows of at most W groups each, a row in the W lanes from `seg` on (`lane` counts
    // from there); the partial sums then have W / 16 terms instead of four, the missing ones being the +0 of above.
    // wave_row: the wave's first row, of `rows`.
    template <int W = 64>
    __device__ __forceinline__ float prepare(int64_t row, int64_t wave_row, int64_t rows, int lane, int groups, int64_t cols, float (&first)[32],
                                             int seg) const {
        // slot 64 i + wlane is piece `piece` of the group of lane 8 i + wlane / 8: group `sub` + 8 i of the row that 8 i / W picks (uniform).
        // Slots past the row's end are filled from its last group: no branch between the requests.
        const int wlane = seg + lane, sub = wlane >> 3, piece = (wlane & 7) ^ sub;
        float acc = 0.0f;
        for (int base = 0; base < groups; base += 64) {
            const int g = base + lane;
            float s = 0.0f;
            if constexpr (kStaged) {
                v4 raw[8];
                const auto group_of = [&](int i) { return base + 8 * i % W + sub; };
                const auto row_of = [&](int i) { const int64_t r = wave_row + 8 * i / W; return (r < rows ? r : rows - 1) * cols; };
                // the lane's element as a 32-bit offset from its row's (uniform) start: one register a slot instead of an address per tensor
                const auto at = [&](int i) { const int gg = group_of(i); return (uint32_t)((gg < groups ? gg : groups - 1) * 32 + piece * 4); };
                const auto piece_at = [&](auto* t, int i) {   // of four elements
                    using V = std::conditional_t<sizeof(*t) == 4, v4, w2>;
                    using B = std::conditional_t<std::is_const_v<std::remove_pointer_t<decltype(t)>>, const char, char>;
                    return reinterpret_cast<std::conditional_t<std::is_const_v<B>, const V, V>*>(reinterpret_cast<B*>(t + row_of(i)) + at(i) * (uint32_t)sizeof(*t));
                };
#pragma unroll
                for (int i = 0; i < 8; ++i) raw[i] = *piece_at(x, i);
                if constexpr (kAdd) {
                    if constexpr (sizeof(TAdd) == 2) {
                        w2 more[8];
#pragma unroll
                        for (int i = 0; i < 8; ++i) more[i] = *piece_at(add, i);
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            raw[i] = raw[i] + v4{u2f(more[i][0] << 16), u2f(more[i][0] & 0xffff0000u), u2f(more[i][1] << 16), u2f(more[i][1] & 0xffff0000u)};
                    } else {
#pragma unroll
                        for (int i = 0; i < 8; ++i) raw[i] = raw[i] + *piece_at(add, i);
                    }
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (group_of(i) < groups) *piece_at(xsum, i) = raw[i];
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) area()[64 * i + wlane] = raw[i];
                wave_settle();
            }
            if (g < groups) {
                float v[32];
                if constexpr (kStaged) read_group(wlane, v);
                else load_group<T>(x + row * cols + g * 32, v);
                if (base == 0) {
#pragma unroll
                    for (int i = 0; i < 32; ++i) first[i] = v[i];
                }
#pragma unroll
                for (int i = 0; i < 32; ++i) v[i] = v[i] * v[i];
                s = tree_sum32(v);
            }
            if constexpr (kStaged) wave_settle();   // the next pass over the row, or the gain, reuses the area
#pragma unroll
            for (int k = 0; k < W / 16; ++k) acc = acc + __shfl(s, seg + (lane & 15) + 16 * k, 64);
        }
        v4 gains[W / 8];
        if constexpr (kStaged) {   // not before: 32 registers that the row needs
#pragma unroll
            for (int i = 0; i < W / 8; ++i) {
                const int gg = 8 * i + sub < groups ? 8 * i + sub : groups - 1;
                gains[i] = *reinterpret_cast<const v4*>(gain + gg * 32 + piece * 4);
            }
        }
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) acc = acc + __shfl_xor(acc, m, 64);
        const float f = 1.0f / __builtin_sqrtf(acc / (float)cols + eps);
        if (lane == 0) factor[row] = f;
        if constexpr (kStaged) {   // the gain of the lanes' first groups, for load()
#pragma unroll
            for (int i = 0; i < W / 8; ++i)
                area()[64 * i + wlane] = gains[i];
            wave_settle();
        }
        return f;
    }
    template <int W>
    __device__ __forceinline__ void stage(int64_t, int64_t, int, int, int64_t, int) const {}
    // v holds the group's raw elements on entry when have_raw
    __device__ __forceinline__ void load(int64_t row, int g, int64_t cols, float f, bool have_raw, float (&v)[32]) const {
        // with a residual sum: what the wave stored in prepare()
        if (!have_raw) load_group<T>((kAdd ? xsum : x) + row * cols + g * 32, v);
#pragma unroll
        for (int i = 0; i < 32; ++i) v[i] = v[i] * f;
        if constexpr (sizeof(T) == 2) {  // .type_as(x)
#pragma unroll
            for (int i = 0; i < 32; i += 2) round_pair_to_bf16(v[i], v[i + 1]);
        }
        float w[32];
        if (kStaged && have_raw) read_group(g, w);
        else load_group<float>(gain + g * 32, w);
#pragma unroll
        for (int i = 0; i < 32; ++i) v[i] = v[i] * w[i];
    }
};

__global__ void silu_of_bf16_kernel(uint16_t* __restrict__ out) {
    const uint32_t x = blockIdx.x * 256 + threadIdx.x;
    out[x] = f32_to_bf16(silu_of_bf16(u2f(x << 16)));
}

template <typename T>
struct SwiGluProducer {
    static constexpr int kOutDtype = sizeof(T) == 2 ? BF16 : F32;
    // bf16: whole lines through 8 KiB of LDS per wave, as in the RMSNorm producer; a group is four pieces here, slot
    // 4 l + (q ^ l / 4 % 4) holds piece q of lane l's group.  Inputs cycled through memory: 16384 x 4096 73 -> 65 us (4.8 TB/s; 76
    // inside a layer's step), 32768 x 4096 141 -> 125; 16384 x 1536 33 either way, up to
    // 4096 x 1728 (11 us) latency
    static constexpr bool kStaged = sizeof(T) == 2, kWithWeight = sizeof(T) == 2;
    static constexpr int kLds = kStaged ? 4 * 512 * 16 : 0;
    const T* h12;  // [rows, 2 cols]: up, then gate

    typedef uint32_t v4 __attribute__((ext_vector_type(4)));
    __device__ __forceinline__ static v4* area() { return reinterpret_cast<v4*>(job_lds) + (threadIdx.x >> 6) * 512; }
    template <int W = 64>
    __device__ __forceinline__ float prepare(int64_t, int64_t, int64_t, int, int, int64_t, float (&)[32], int) const { return 0.0f; }
    // every lane of the wave: the groups base + lane of its rows
    template <int W>
    __device__ __forceinline__ void stage(int64_t wave_row, int64_t rows, int base, int groups, int64_t cols, int wlane) const {
        if constexpr (kStaged) {
            const int sub = wlane >> 2, piece = (wlane & 3) ^ ((wlane >> 4) & 3);
            v4 up[4], gate[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t r = wave_row + 16 * i / W;
                const int g = base + 16 * i % W + sub;
                const T* at = h12 + (r < rows ? r : rows - 1) * 2 * cols + (g < groups ? g : groups - 1) * 32 + piece * 8;
                up[i] = *reinterpret_cast<const v4*>(at);
                gate[i] = *reinterpret_cast<const v4*>(at + cols);
            }
            wave_settle();   // the lanes have read the groups before
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                area()[64 * i + wlane] = up[i];
                area()[256 + 64 * i + wlane] = gate[i];
            }
            wave_settle();
        }
    }
    __device__ __forceinline__ static void read_group(int half, float (&v)[32]) {
        const int wlane = threadIdx.x & 63;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const v4 t = area()[256 * half + 4 * wlane + (q ^ ((wlane >> 2) & 3))];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[8 * q + 2 * e] = u2f(t[e] << 16);
                v[8 * q + 2 * e + 1] = u2f(t[e] & 0xffff0000u);
            }
        }
    }
    __device__ __forceinline__ void load(int64_t row, int g, int64_t cols, float, bool, float (&v)[32]) const {
        float gate[32];
        if constexpr (kStaged) {
            read_group(0, v);
            read_group(1, gate);
        } else {
            load_group<T>(h12 + row * 2 * cols + g * 32, v);
            load_group<T>(h12 + row * 2 * cols + cols + g * 32, gate);
        }
        if constexpr (sizeof(T) == 2) {
            swiglu_group_bf16(v, gate);
        } else {
#pragma unroll
            for (int i = 0; i < 32; ++i) v[i] = silu_fixed(v[i]) * gate[i];
        }
    }
};

// quest RTN + clip mask (the forward quantizer) of rows that a producer computes
// W: lanes per row (64, or 32 / 16 for rows of at most that many groups: two / four rows per wave)
template <typename P, bool TILED, int W = 64>
struct ProducedRowsJob {
    static constexpr int kLds = P::kLds;
    static constexpr int kWaves = 1;
    P prod;
    int64_t rows, cols;
    float c;
    uint32_t sign_word;
    GroupOut out;
    unsigned blocks;

    ProducedRowsJob(const P& prod_, int64_t rows_, int64_t cols_, uint32_t sign_word_, const GroupOut& out_)
        : prod(prod_), rows(rows_), cols(cols_), c(hadamard_scale(32, P::kOutDtype)), sign_word(sign_word_), out(out_),
          blocks((unsigned)((rows_ + 4 * (64 / W) - 1) / (4 * (64 / W)))) {}

    __device__ __forceinline__ void run(unsigned bid) const {
        const int wlane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int lane = wlane & (W - 1), seg = wlane - lane;  // place in the row's segment of the wave
        const int64_t wave_row = ((int64_t)bid * 4 + __builtin_amdgcn_readfirstlane(wave)) * (64 / W);
        int64_t row = wave_row + seg / W;
        if (wave_row >= rows) return;  // a whole wave
        if (row >= rows) row = rows - 1;    // a segment past the end repeats the last row: same values to the same places
        const int groups = (int)(cols / 32);
        float v[32];
        const float state = prod.template prepare<W>(row, wave_row, rows, lane, groups, cols, v, seg);
        // TILED: the row's groups padded to a multiple of four with zero codes and scales; the padding lanes of the last quad
        // are inactive in the loop, so that the scale gather reads zeros from them
        const int groups_p = TILED ? (groups + 3) & ~3 : groups;
        const auto tile_slot = [&](int g) { return (row >> 4) * 16 * groups_p + ((g >> 2) * 64 + (int)(row & 15) * 4 + (g & 3)); };
        for (int base = 0; base < groups; base += W) {
            const int g = base + lane;
            prod.template stage<W>(wave_row, rows, base, groups, cols, wlane);
            if (g >= groups) continue;
            const int64_t gi = row * groups + g;
            const int64_t ci = TILED ? tile_slot(g) : gi;
            prod.load(row, g, cols, state, g == lane, v);
            rotate_group(v, c, sign_word);
            GroupCodes o;
            quantize_group_regs<QUEST_RTN, true>(v, 0, gi, o);
            out.codes[ci] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
            if constexpr (TILED) {
                const uint32_t s1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o.scale_byte, 0x55, 0xf, 0xf, false);
                const uint32_t s2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o.scale_byte, 0xAA, 0xf, 0xf, false);
                const uint32_t s3 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o.scale_byte, 0xFF, 0xf, 0xf, false);
                if ((lane & 3) == 0)
                    *reinterpret_cast<uint32_t*>(out.scales + row * groups_p + g) = o.scale_byte | (s1 << 8) | (s2 << 16) | (s3 << 24);
            } else {
                out.scales[gi] = (uint8_t)o.scale_byte;
            }
            out.maskbits[gi] = o.keep;
        }
        if (TILED && lane < groups_p - groups) out.codes[tile_slot(groups + lane)] = make_uint4(0u, 0u, 0u, 0u);
    }
};

// RMSNorm and quantizer with eight elements to a lane, four lanes to a group: fp32 rows of at most 2048 elements, tiled codes.  The same operations in
// the same order as RmsNormProducer and quantize_group_regs, sums of a group's or a row's parts by lane exchanges instead of in one lane's registers:
// the same bits.  A workgroup has as many rows as fit, each in a whole number of sixteen lanes (four groups, whose scale bytes leave together); one
// barrier, behind the groups' sums of squares.  With a group to a lane, 4096 rows of 640 are 2048 waves of 1400 instructions with 20 of every 32
// lanes at work; here 5500 waves of 300.  What bounds it at such sizes is latency, and with a summand the sum's way to memory: 4096 x 640 in an
// evaluated 30 M model 11.1 -> 9.7 us, a pass of it 847 -> 836; past the caches the sum is no faster.  Sizes: octets_serve().
template <typename TA>
struct RmsNormOctetsJob {
    static constexpr int kLds = 256;   // a workgroup's group sums, at most 64
    static constexpr int kWaves = 0;
    static constexpr bool kAdd = !std::is_void<TA>::value;
    using TAdd = typename std::conditional<kAdd, TA, float>::type;
    RmsNormProducer<float, TA> prod;
    int64_t rows, cols;
    float c;
    uint32_t sign_word;
    GroupOut out;
    int groups, groups_p, wg_rows;
    unsigned blocks;

    RmsNormOctetsJob(const RmsNormProducer<float, TA>& prod_, int64_t rows_, int64_t cols_, uint32_t sign_word_, const GroupOut& out_)
        : prod(prod_), rows(rows_), cols(cols_), c(hadamard_scale(32, F32)), sign_word(sign_word_), out(out_), groups((int)(cols_ / 32)),
          groups_p((groups + 3) & ~3), wg_rows(256 / (groups_p * 4)), blocks((unsigned)((rows_ + wg_rows - 1) / wg_rows)) {}

    // the sum over a group's four lanes of what are sums of eight neighbours each: the upper levels of its pairwise tree
    __device__ __forceinline__ static float over_group(float v) {
        v = v + lane_xor<1>(v);
        return v + lane_xor<2>(v);
    }
    __device__ __forceinline__ static float tree_sum8(const float (&p)[8]) { return ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])); }

    __device__ __forceinline__ void run(unsigned bid) const {
        typedef float v4 __attribute__((ext_vector_type(4)));
        float* sums = reinterpret_cast<float*>(job_lds);   // [row of the workgroup][group]
        const int tid = threadIdx.x, lane = tid & 63, per_row = groups_p * 4;
        const int r = tid / per_row, at = tid - r * per_row, g = at >> 2, octet = at & 3;
        const int64_t row = (int64_t)bid * wg_rows + r;
        const bool in_row = r < wg_rows && row < rows, mine = in_row && g < groups;
        float v[8], gain[8];
        const int64_t first = row * cols + g * 32 + octet * 8;
        float s = 0.0f;
        if (mine) {
            const v4* src = reinterpret_cast<const v4*>(prod.x + first);
            v4 lo = src[0], hi = src[1];
            const v4* gp = reinterpret_cast<const v4*>(prod.gain + g * 32 + octet * 8);
            const v4 g0 = gp[0], g1 = gp[1];
            if constexpr (kAdd) {
                if constexpr (sizeof(TAdd) == 2) {
                    const uint4 m = *reinterpret_cast<const uint4*>(prod.add + first);
                    lo = lo + v4{u2f(m.x << 16), u2f(m.x & 0xffff0000u), u2f(m.y << 16), u2f(m.y & 0xffff0000u)};
                    hi = hi + v4{u2f(m.z << 16), u2f(m.z & 0xffff0000u), u2f(m.w << 16), u2f(m.w & 0xffff0000u)};
                } else {
                    const v4* m = reinterpret_cast<const v4*>(prod.add + first);
                    lo = lo + m[0];
                    hi = hi + m[1];
                }
                v4* dst = reinterpret_cast<v4*>(prod.xsum + first);
                dst[0] = lo;
                dst[1] = hi;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = lo[e];
                v[4 + e] = hi[e];
                gain[e] = g0[e];
                gain[4 + e] = g1[e];
            }
            float sq[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) sq[e] = v[e] * v[e];
            s = tree_sum8(sq);
        }
        job_requests_issued();
        s = over_group(s);
        if (mine && octet == 0) sums[r * groups_p + g] = s;
        __syncthreads();
        // The row's sum as RmsNormProducer orders it: sixteen partial sums of every sixteenth group, then pairwise.  A wave's lanes are of at most
        // four rows: sixteen lanes add up each of them.
        const int r0 = (tid - lane) / per_row;
        float total;
        {
            const int rr = r0 + (lane >> 4);
            float acc = 0.0f;
            if (rr < wg_rows)
                for (int j = lane & 15; j < groups; j += 16) acc = acc + sums[rr * groups_p + j];
#pragma unroll
            for (int m = 1; m < 16; m <<= 1) acc = acc + __shfl_xor(acc, m, 64);
            total = acc;
        }
        const float f = __shfl(1.0f / __builtin_sqrtf(total / (float)cols + prod.eps), (r - r0) * 16, 64);
        if (!in_row) return;
        if (at == 0) prod.factor[row] = f;
        const int64_t ci = ((row >> 4) * 16 * groups_p + ((g >> 2) * 64 + (int)(row & 15) * 4 + (g & 3))) * 4 + octet;
        uint32_t* codes = reinterpret_cast<uint32_t*>(out.codes);
        uint32_t word = 0u, scale_byte = 0u;
        if (mine) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = v[e] * f * gain[e];
#pragma unroll
            for (int h = 1; h < 8; h <<= 1)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (i & h) continue;
                    const float a = v[i], b = v[i + h];
                    v[i] = a + b;
                    v[i + h] = a - b;
                }
            octet_cross_lane_stage<1>(v, octet);
            octet_cross_lane_stage<2>(v, octet);
            const uint32_t signs = sign_word >> (8 * octet);
            float sq[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = v[e] * u2f(f2u(-c) ^ (((signs >> e) & 1u) << 31));
                sq[e] = v[e] * v[e];
            }
            const float ms = over_group(tree_sum8(sq)) * 0.03125f, m = over_group(tree_sum8(v)) * 0.03125f;
            float var = ms - m * m;
            var = var > 0.0f ? var : 0.0f;
            int E = (int)((f2u(kQuestG * __builtin_sqrtf(var) + 1e-8f) >> 23) & 0xffu) - 127;
            E = E > 127 ? 127 : E;
            scale_byte = (uint32_t)(E + 127);
            const float hw_scale = pow2i(E), thr = 6.0f * hw_scale;
            uint32_t keep = 0u;
#pragma unroll
            for (int e = 7; e >= 0; --e) keep = __builtin_amdgcn_alignbit(keep, f2u(fabsf(v[e]) - thr), 31);
            const auto convert = [&](auto below) {
                word = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, below(v[0]), below(v[1]), hw_scale, 0);
                word = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, below(v[2]), below(v[3]), hw_scale, 1);
                word = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, below(v[4]), below(v[5]), hw_scale, 2);
                word = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, below(v[6]), below(v[7]), hw_scale, 3) ^ 0x88888888u;
            };
            if (__builtin_expect(ms < __builtin_inff(), 1)) convert([](float x) { return below_ties(x); });
            else convert([](float x) { return below_ties_any(x); });
            reinterpret_cast<uint8_t*>(out.maskbits)[(row * groups + g) * 4 + octet] = (uint8_t)keep;
        }
        job_stores_next();
        codes[ci] = word;   // zeros in the padding groups
        // a row's lanes of four groups are sixteen aligned ones: their scale bytes in one dword
        uint32_t four = scale_byte << (8 * (g & 3));
        four |= f2u(lane_xor<4>(u2f(four)));
        four |= f2u(lane_xor<8>(u2f(four)));
        if ((at & 15) == 0) *reinterpret_cast<uint32_t*>(out.scales + row * groups_p + g) = four;
    }
};

// The quantizer of the layer's weight rides in the same grid, behind the rows, where the launch is one of a training step under
// autocast: fp32 weights, tiled codes of any extents.  By itself it is a launch of a few microseconds that mostly starts and ends
// (1536 x 4096: 9.6 us, 4608 x 1536 11).  us per training step with the two launches and with one: 16384 x 1536 x 4608 behind its norm 449 ->
// 443.5, 16384 x 4096 x 1536 behind SwiGLU 431 -> 424.5, 1024 x 4096 x 8192 201.7 -> 198.4.
using WeightJob = RowmajorTiledJob<float, QUEST_RTN, true, 32, true>;
WeightJob weight_job(const RowmajorArgs& w) {
    return WeightJob(w.x, w.rows, w.cols, make_rotation<32>(w.dtype, w.signs), 0,
                     GroupOut{reinterpret_cast<uint4*>(w.codes), w.scales, reinterpret_cast<uint32_t*>(w.maskbits), nullptr});
}

template <typename P, int W>
void launch_produced_w(const P& prod, int64_t rows, int64_t cols, uint32_t sign_word, const GroupOut& out, bool tiled, const RowmajorArgs* weight,
                       hipStream_t stream) {
    const ProducedRowsJob<P, true, W> job(prod, rows, cols, sign_word, out);
    if constexpr (P::kWithWeight)
        if (weight) return launch_jobs(stream, job, weight_job(*weight));
    if (tiled) launch_job(job, stream);
    else launch_job(ProducedRowsJob<P, false, W>(prod, rows, cols, sign_word, out), stream);
}

template <typename P>
void launch_produced(const P& prod, int64_t rows, int64_t cols, uint32_t sign_word, uint8_t* codes, uint8_t* scales,
                     uint8_t* maskbits, bool tiled, const RowmajorArgs* weight, hipStream_t stream) {
    const GroupOut out{reinterpret_cast<uint4*>(codes), scales, reinterpret_cast<uint32_t*>(maskbits), nullptr};
    if (cols <= 16 * 32) launch_produced_w<P, 16>(prod, rows, cols, sign_word, out, tiled, weight, stream);
    else if (cols <= 32 * 32) launch_produced_w<P, 32>(prod, rows, cols, sign_word, out, tiled, weight, stream);
    else launch_produced_w<P, 64>(prod, rows, cols, sign_word, out, tiled, weight, stream);
}

}  // namespace

namespace {
// Where RmsNormOctetsJob is the faster one: a row fits a workgroup, and the tensor is small enough for waves to be what is missing.  us behind a copy
// with a bf16 summand, a group and an octet to a lane: 8192 x 640 14.3 and 12.7, 16384 x 640 22.9 and 20.9, 4096 x 1536 15.7 and 13.7, 8192 x 1536 25.8 and 22.7,
// 8192 x 2048 30.9 and 30.2; where the line lies 16384 x 1024 29.9 and 30.0, 16384 x 1536 57.7 either way, 32768 x 1536 102.6 and 105.8.
bool octets_serve(int64_t rows, int64_t cols) { return cols <= 2048 && rows * cols <= 1 << 24; }
}  // namespace
bool producer_takes_weight(int dtype, int add_dtype, int w_dtype) { return dtype == F32 && add_dtype == BF16 && w_dtype == F32; }
bool swiglu_takes_weight(int dtype, int w_dtype) { return dtype == BF16 && w_dtype == F32; }

// Q(rmsnorm(x) * gain): Hadamard block 32, quest RTN, clip mask; factor [rows] receives 1 / sqrt(mean(x^2) + eps).
// add != null (x fp32 only): the norm's input is x + add, also written to xsum [rows, cols] fp32.
hipError_t rmsnorm_quantize_hd32(const void* x, int dtype, const void* add, int add_dtype, void* xsum, const float* gain, float eps,
                                 int64_t rows, int64_t cols, uint32_t sign_word, uint8_t* codes, uint8_t* scales, uint8_t* maskbits,
                                 float* factor, bool tiled, const RowmajorArgs* weight, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    if (weight && !(tiled && producer_takes_weight(dtype, add ? add_dtype : BF16, weight->dtype))) return hipErrorInvalidValue;
    if (tiled && dtype == F32 && octets_serve(rows, cols)) {
        const float* xp = reinterpret_cast<const float*>(x);
        float* sp = reinterpret_cast<float*>(xsum);
        const GroupOut out{reinterpret_cast<uint4*>(codes), scales, reinterpret_cast<uint32_t*>(maskbits), nullptr};
        const auto go = [&](const auto* summand) {
            using TA = std::remove_const_t<std::remove_pointer_t<decltype(summand)>>;
            const RmsNormOctetsJob<TA> job({xp, gain, factor, eps, reinterpret_cast<const typename RmsNormOctetsJob<TA>::TAdd*>(summand), sp}, rows, cols, sign_word, out);
            if constexpr (!std::is_same<TA, float>::value)
                if (weight) return launch_jobs(stream, job, weight_job(*weight));
            launch_job(job, stream);
        };
        if (!add) go(static_cast<const void*>(nullptr));
        else if (add_dtype == BF16) go(static_cast<const uint16_t*>(add));
        else go(static_cast<const float*>(add));
        return hipGetLastError();
    }
    if (add) {
        if (dtype != F32) return hipErrorInvalidValue;
        const float* xp = reinterpret_cast<const float*>(x);
        float* sp = reinterpret_cast<float*>(xsum);
        if (add_dtype == BF16)
            launch_produced(RmsNormProducer<float, uint16_t>{xp, gain, factor, eps, reinterpret_cast<const uint16_t*>(add), sp}, rows,
                            cols, sign_word, codes, scales, maskbits, tiled, weight, stream);
        else
            launch_produced(RmsNormProducer<float, float>{xp, gain, factor, eps, reinterpret_cast<const float*>(add), sp}, rows, cols,
                            sign_word, codes, scales, maskbits, tiled, weight, stream);
    } else if (dtype == BF16) {
        launch_produced(RmsNormProducer<uint16_t>{reinterpret_cast<const uint16_t*>(x), gain, factor, eps, nullptr, nullptr}, rows,
                        cols, sign_word, codes, scales, maskbits, tiled, weight, stream);
    } else {
        launch_produced(RmsNormProducer<float>{reinterpret_cast<const float*>(x), gain, factor, eps, nullptr, nullptr}, rows, cols,
                        sign_word, codes, scales, maskbits, tiled, weight, stream);
    }
    return hipGetLastError();
}

// the bf16 silu of every bf16 bit pattern, 65536 values
hipError_t silu_of_bf16_table(uint16_t* out, hipStream_t stream) {
    silu_of_bf16_kernel<<<dim3(256), dim3(256), 0, stream>>>(out);
    return hipGetLastError();
}

// Q(silu(up) * gate) of h12 [rows, 2 hidden] = (up, gate): Hadamard block 32, quest RTN, clip mask
hipError_t swiglu_quantize_hd32(const void* h12, int dtype, int64_t rows, int64_t hidden, uint32_t sign_word,
                                uint8_t* codes, uint8_t* scales, uint8_t* maskbits, bool tiled, const RowmajorArgs* weight, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    if (weight && !(tiled && swiglu_takes_weight(dtype, weight->dtype))) return hipErrorInvalidValue;
    if (dtype == BF16)
        launch_produced(SwiGluProducer<uint16_t>{reinterpret_cast<const uint16_t*>(h12)}, rows, hidden, sign_word, codes,
                        scales, maskbits, tiled, weight, stream);
    else
        launch_produced(SwiGluProducer<float>{reinterpret_cast<const float*>(h12)}, rows, hidden, sign_word, codes, scales,
                        maskbits, tiled, weight, stream);
    return hipGetLastError();
}

// ---- the quantizer launches of one layer, and of a quantizer module -----------------------------------------------

namespace {
template <typename F>
void with_mode(int mode, F&& f) {
    switch (mode) {
        case QUEST_RTN: return f(std::integral_constant<int, QUEST_RTN>{});
        case ABSMAX_RTN: return f(std::integral_constant<int, ABSMAX_RTN>{});
        case ABSMAX_SR: return f(std::integral_constant<int, ABSMAX_SR>{});
        default: return f(std::integral_constant<int, QUEST_SR>{});
    }
}
template <typename F>
void with_elem_type(int dtype, F&& f) {
    if (dtype == BF16) f(uint16_t{});
    else f(float{});
}
template <typename F>
void with_absmax_mode(int mode, F&& f) {
    if (mode == ABSMAX_SR) f(std::integral_constant<int, ABSMAX_SR>{});
    else f(std::integral_constant<int, ABSMAX_RTN>{});
}
template <typename F>
void with_flag(bool on, F&& f) {
    if (on) f(std::true_type{});
    else f(std::false_type{});
}
template <typename F>
void with_hadamard(int hd, F&& f) {
    if (hd == 32) f(std::integral_constant<int, 32>{});
    else if (hd == 64) f(std::integral_constant<int, 64>{});
    else f(std::integral_constant<int, 128>{});
}
}  // namespace

hipError_t quantize_values(const void* x, int dtype, int64_t rows, int64_t cols, int hd, const SignBits& sb, int mode, uint64_t seed, uint8_t* maskbits,
                           void* values, hipStream_t stream) {
    const int64_t n_groups = rows * cols / 32;
    with_elem_type(dtype, [&](auto t) {
        using T = decltype(t);
        const int64_t bytes = rows * cols * (int64_t)sizeof(T);
        with_mode(mode, [&](auto m) {
            constexpr int MODE = decltype(m)::value;
            const auto go = [&](auto k) {
                with_hadamard(hd, [&](auto h) {
                    constexpr int HD = decltype(h)::value;
                    quantize_values_kernel<T, MODE, decltype(k)::value, HD><<<dim3((unsigned)((n_groups + 255) / 256)), dim3(256), 256 * 32 * sizeof(T), stream>>>(
                        reinterpret_cast<const T*>(x), n_groups, make_rotation<HD>(dtype, sb), seed, reinterpret_cast<uint32_t*>(maskbits), reinterpret_cast<T*>(values),
                        bytes >= kPastTheCaches, bytes >= kMoreThanTheCaches);
                });
            };
            if constexpr (MODE == QUEST_RTN || MODE == QUEST_SR) go(std::true_type{});
            else with_flag(maskbits != nullptr, go);
        });
    });
    return hipGetLastError();
}

hipError_t quantize_layer_forward(const RowmajorArgs& x, const RowmajorArgs* w, int hd, hipStream_t stream) {
    const auto out_of = [](const RowmajorArgs& a) {
        return GroupOut{reinterpret_cast<uint4*>(a.codes), a.scales, reinterpret_cast<uint32_t*>(a.maskbits), nullptr};
    };
    const auto ragged = [](const RowmajorArgs& a) { return a.rows % 16 != 0 || a.cols % 128 != 0; };
    with_hadamard(hd, [&](auto h) {
        with_flag(ragged(x) || (w && ragged(*w)), [&](auto p) {
            constexpr int HD = decltype(h)::value;
            const auto job_of = [&](const RowmajorArgs& a, auto t) {
                return RowmajorTiledJob<decltype(t), QUEST_RTN, true, HD, decltype(p)::value>(a.x, a.rows, a.cols, make_rotation<HD>(a.dtype, a.signs),
                                                                                              0, out_of(a));
            };
            with_elem_type(x.dtype, [&](auto tx) {
                if (!w) launch_jobs(stream, job_of(x, tx));
                else with_elem_type(w->dtype, [&](auto tw) { launch_jobs(stream, job_of(x, tx), job_of(*w, tw)); });
            });
        });
    });
    return hipGetLastError();
}

namespace {
// the two quantizations of e as jobs (with `more` jobs' instantiations for the same mode, Hadamard block and raggedness in one grid)
template <typename F>
hipError_t with_error_jobs(const ErrorArgs& a, int hd, const SignBits& signs, int mode, const uint64_t* seed_base, bool ragged, F&& f) {
    const GroupOut orow{reinterpret_cast<uint4*>(a.codes_rows), a.scales_rows, nullptr, nullptr};
    with_absmax_mode(mode, [&](auto m) {
        with_hadamard(hd, [&](auto h) {
            constexpr int M = decltype(m)::value, HD = decltype(h)::value;
            with_elem_type(a.dtype, [&](auto t) {
                with_flag(ragged, [&](auto p) {
                    using T_ = decltype(t);
                    constexpr bool PADDED = decltype(p)::value;
                    const Rotation rot = make_rotation<HD>(a.dtype, signs);
                    TransposedJob<T_, M, false, HD, PADDED> jt(a.e, a.T, a.O, rot, a.seed_transposed, a.codes_transposed, a.scales_transposed, nullptr, true);
                    RowmajorTiledJob<T_, M, false, HD, PADDED> jr(a.e, a.T, a.O, rot, a.seed_rows, orow);
                    jt.seed_base = jr.seed_base = seed_base;
                    f(jt, jr, m, h, p);
                });
            });
        });
    });
    return hipGetLastError();
}
bool ragged_extents(int64_t a, int64_t b) { return a % 128 != 0 || b % 128 != 0; }
}  // namespace

hipError_t quantize_error(const ErrorArgs& e, int hd, const SignBits& signs, int mode, const E5m2Args& x, const E5m2Args& w, hipStream_t stream) {
    return with_error_jobs(e, hd, signs, mode, nullptr, ragged_extents(e.T, e.O),
                           [&](const auto& jt, const auto& jr, auto, auto, auto) { launch_jobs(stream, SpanJob(x), SpanJob(w), jt, jr); });
}

hipError_t quantize_layer_backward(const ErrorArgs& e, int hd, const SignBits& signs, int mode, const RequantArgs& x, const RequantArgs& w,
                                   const uint64_t* seed_base, hipStream_t stream) {
    return with_error_jobs(e, hd, signs, mode, seed_base, ragged_extents(e.T, e.O) || ragged_extents(x.R, x.C) || ragged_extents(w.R, w.C),
                           [&](const auto& jt, const auto& jr, auto m, auto h, auto p) {
        using Requant = RequantTiledJob<decltype(m)::value, decltype(h)::value, decltype(p)::value>;
        // The longest workgroups first (four groups a lane, two, one): what starts last is what ends soonest.  us per training step with the error signal's
        // first, as the operands' used to wait behind it, and so: 16480 x 1728 x 640 112.4 -> 102.3, 4096 x 2048^2 68.4 -> 62.2, 2048 x 4096^2 106.6 -> 98.0, blocks
        // of 128 8192 x 1536 x 4608 176.6 -> 169.1, 16384 x 1536 x 4608 behind its norm 419.9 -> 405.7, 8192 x 4096^2 271.7 -> 268.7, 8192 x 4096 x 11008 679.1 ->
        // 677.2; only x first 0 to 7 % slower than this, the rows of e ahead of its columns 0 to 5 %.
        launch_jobs(stream, Requant(x, signs, seed_base), Requant(w, signs, seed_base), jt, jr);
    });
}

}  // namespace qm
