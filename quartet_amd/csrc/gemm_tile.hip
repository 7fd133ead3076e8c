// FP4 x FP4 "TN" product on tiles from 64 x 32 to 256 x 128: everything that the persistent 256 x 256 kernel of gemm.hip
// is too coarse for -- short contractions, matrices with few tiles, and any number of rows and (multiples of eight) columns.
//
// One design, five tile shapes.  A workgroup of W waves owns a BM x BN tile, each wave WM x WN of it in 32 x 32 blocks of
// v_mfma_scale_f32_32x32x64_f8f6f4.  Operands go global -> LDS directly (16 bytes per lane, XOR-swizzled 16-byte slots)
// into a ring of STAGES K steps of 128, scales beside them in blocks of four steps; one barrier per step.  Rows past the end of a
// matrix are requested as its last row (their products are dropped), so no request leaves the operands.  bf16 results pass
// through the ring's LDS and leave as 16-byte pieces of whole rows; on that way a lane holds eight consecutive columns,
// which is what the masked inverse Hadamard rotation of the layer's backward pass works on: it is applied there (blocks of
// 32, 64 or 128 along N), with the arithmetic of the stand-alone kernel, bit for bit, and the rotated-basis gradient never
// travels through memory.
//
// What bounds it: at 256 x 128 the LDS reads of the K loop (1.5 x the 256 x 256 kernel's bytes per flop) and, for short
// contractions, the tile boundary, which the neighbour workgroup on the same CU covers; the smaller tiles are latency-bound
// and exist to put more workgroups on the chip.  Accumulation order over K is the same in every shape and in gemm.hip's
// kernels: results depend on the choice only where a product is cut into K ranges.  (gemm_rows.hip's order is its own.)
//
// The same kernel multiplies FP4 with a B of six (E3M2) or eight (E5M2) bits, which is how the error-only scheme contracts over
// the rows of a packed operand (expand.hip): 1.5 times the bytes of B at FP4's matrix rate, or twice the bytes at half of it.  4096^3
// among the other kernels of a training step, 8 waves of 128 x 64 on 256 x 256, rotation included: 50 us in six bits, 63 in eight,
// where the FP4 x bf16 kernel (gemm_fp4_bf16.hip) takes 113 us and more.  4 waves of 128 x 128 read a third fewer bytes from LDS and
// took 67 where these took 58 (with the rotation as it was then, see rotate_rows).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gemm_common.h"
#include "hadamard_octet.h"
#include "quantize_group.h"

namespace qm {

namespace {

// E5M2_B: B is eight bits wide (expand.hip), two 1 KiB blocks of 64 contraction indices per 16 columns and K step.
// BLOCKS: scales travel in blocks of four K steps, 16 bytes per row and request, into an area of their own, from where every wave
// takes its rows' into registers (K >= 512 and 4-byte aligned scale rows).  Otherwise one dword per row and K step, in the ring:
// every dword lies in another line, and those requests are two thirds of all.  4608 x 1536 x 8192 55 -> 40 us,
// 2048 x 4096 x 4096 32 -> 25, 512 x 11008 x 4096 27 -> 22; without any scale requests (wrong results) 37, 22 and 19.
template <int BM_, int BN_, int WM_, int WN_, int STAGES_, int OCC_, bool E5M2_B = false, bool BLOCKS_ = true, bool MIXED_ = false>
struct TileShape {
    using Narrow = TileShape<BM_, BN_, WM_, WN_, STAGES_, OCC_, E5M2_B, false>;
    using Mixed = TileShape<BM_, BN_, WM_, WN_, STAGES_, OCC_, true, true, true>;
    static constexpr bool kBlocks = BLOCKS_;
    static constexpr bool kWideB = E5M2_B;
    static constexpr bool kMixed = MIXED_;   // blocks of four K steps and 256 columns of B in six or eight bits each
    static constexpr int kBBlocks = E5M2_B ? 2 : 1;
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, STAGES = STAGES_, OCC = OCC_;   // OCC: workgroups per CU
    static constexpr int kWavesN = BN / WN, kWaves = (BM / WM) * kWavesN, kThreads = kWaves * 64;
    static constexpr int TM = WM / 32, TN = WN / 32;
    static constexpr int kALoads = BM / 16 / kWaves, kBLoads = BN / 16 * kBBlocks / kWaves;   // 1 KiB wave-loads per wave and K step
    static constexpr int kUnits6 = BN / 16 + BN / 32, kBLoads6 = (kUnits6 + kWaves - 1) / kWaves;   // six-bit B
    static constexpr int kAUnits = (BM + 63) / 64, kUnits = kAUnits + (BN + 63) / 64;   // requests of 64 rows' scales each
    static constexpr int kSLoads = (kUnits + kWaves - 1) / kWaves;
    static constexpr int kLoads = kALoads + kBLoads + (kBlocks ? 0 : kSLoads);   // requests per wave and K step
    static constexpr int kUnitBytes = kBlocks ? 1024 : 256;
    // scales: in the stage (BLOCKS: behind the ring)
    static constexpr int kBOff = BM * kRowBytes, kCodeBytes = (BM + BN * kBBlocks) * kRowBytes;
    static constexpr int kStageBytes = kCodeBytes + (kBlocks ? 0 : kUnits * kUnitBytes);
    static constexpr int kSAOff = kBlocks ? STAGES * kStageBytes : kCodeBytes, kSBOff = kSAOff + kAUnits * kUnitBytes;
    static constexpr int kFlagOff = STAGES * kStageBytes + (kBlocks ? kUnits * kUnitBytes : 0);
    static constexpr int kRingBytes = kFlagOff + (kMixed ? kMaxSixBlocks / 8 : 0);
    static constexpr int kMUnits = BM * BN / 2048, kMLoads = (kMUnits + kWaves - 1) / kWaves;   // mask words of the tile, 64 at a time
    // ahead of the operands where there is room beside the ring for OCC workgroups per CU
    static constexpr bool kMaskEarly = BM < 256 && (kRingBytes + kMUnits * 256) * OCC <= 160 * 1024;
    static constexpr int kPitch = BN * 2 + 16;                   // bytes per staged row of the bf16 tile
    static constexpr int kChunks = BN / 8;                       // 16-byte pieces per row
    static constexpr int kRowsPerPass = kThreads / kChunks, kPasses = BM / kRowsPerPass;
    static_assert(kALoads * 16 * kWaves == BM && kBLoads * 16 * kWaves == BN * kBBlocks, "whole wave-loads per wave");
    static constexpr int kMaskOff = kMaskEarly ? kRingBytes : (BM * kPitch + 255) / 256 * 256;
    static constexpr int kSmemBytes = kMaskOff + kMUnits * 256 > kRingBytes ? kMaskOff + kMUnits * 256 : kRingBytes;
    static_assert(kSmemBytes * OCC <= 160 * 1024, "LDS of the resident workgroups");
    static_assert(BM * kPitch <= kMaskOff, "the epilogue stages through the operand ring");
    static_assert(TM == 1 || TM == 2 || TM == 4, "scale dwords of a lane are read as one vector");
    static_assert(TN == 1 || TN == 2, "scale dwords of a lane are read as one vector");
};

template <int N>
__device__ __forceinline__ void read_dwords(const uint8_t* p, uint32_t (&v)[N]) {
    if constexpr (N == 4) {
        const uint4 q = *reinterpret_cast<const uint4*>(p);
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else if constexpr (N == 2) {
        const uint2 q = *reinterpret_cast<const uint2*>(p);
        v[0] = q.x; v[1] = q.y;
    } else {
        v[0] = *reinterpret_cast<const uint32_t*>(p);
    }
}

template <class S>
struct TilePlan {
    const uint8_t* a;   // uniform: first code byte of the tile's panels (K step 0)
    const uint8_t* b;
    const uint8_t* s[S::kSLoads];      // uniform: scale array behind this wave's scale requests
    uint32_t voff_a[S::kALoads];       // this lane's byte offset from it: a row of the wave-load (clamped to the matrix) and
    uint32_t voff_b[S::kBLoads];       //   the swizzled 16-byte column
    uint32_t voff_s[S::kSLoads];
    uint32_t half_back;                // pieces 2 and 3 of a half step re-read pieces 0 and 1
    int kstep_a, kstep_b;              // bytes from one K step to the next: 64 row-major, 1024 tiled
    uint32_t lds_a, lds_b, lds_s[S::kSLoads];   // wave-uniform LDS addresses (stage 0)
};

// half: the step covers only 64 contraction indices (the last step of a K with K % 128 == 64, row-major operands).  Its
// lanes request the row's final two 16-byte pieces in place of all four, and the scale dword that ends with the row's last
// byte (two bytes early), so that no request leaves the row; the consumer shifts that dword down by 16 bits, which puts
// the two real scale bytes first and zeros (2^-127: products vanish) where the missing half of the step would be.
// live: all ones, or zero for a request that nobody reads, whose lanes then all ask for the panel's first sixteen bytes: one line instead of eight
// (and of 64 for scales).  They keep a wave's counts of outstanding requests uniform, STAGES steps and a block of scales at the end of every tile: of K = 640
// a third of all lines.  us per training step with repeats of the last step and now: 16480 x 1728 x 640 107.2 -> 105.2, 16384 x 640 x 1920 113.5 -> 112.3.
template <class S>
__device__ __forceinline__ void tile_issue(const TilePlan<S>& p, int stage, int ks, bool half, uint32_t live = ~0u) {
    const uint32_t off = (uint32_t)stage * S::kStageBytes;
    const uint32_t back = half ? p.half_back : 0u;
    const uint8_t* a = p.a + (int64_t)ks * p.kstep_a;
    const uint8_t* b = p.b + (int64_t)ks * p.kstep_b;
#pragma unroll
    for (int j = 0; j < S::kALoads; ++j) load_lds_b128_s(a, (p.voff_a[j] - back) & live, p.lds_a + off + j * 1024);
#pragma unroll
    for (int j = 0; j < S::kBLoads; ++j) load_lds_b128_s(b, (p.voff_b[j] - back) & live, p.lds_b + off + j * 1024);
    const int sback = half ? 2 : 0;
#pragma unroll
    for (int u = 0; u < S::kSLoads; ++u)
        if constexpr (!S::kBlocks) load_lds_b32_s(p.s[u] + ks * 4 - sback, p.voff_s[u], p.lds_s[u] + off);
}
// BLOCKS: the 16 bytes of every row from K step ks on
template <class S>
__device__ __forceinline__ void tile_issue_scales(const TilePlan<S>& p, int ks, uint32_t live = ~0u) {
#pragma unroll
    for (int u = 0; u < S::kSLoads; ++u) load_lds_b128_s(p.s[u] + ks * 4, p.voff_s[u] & live, p.lds_s[u]);
}
// the scale dwords of a lane's rows for four K steps
template <class S>
struct TileScales {
    uint4 a[S::TM], b[S::TN];
};
template <class S>
__device__ __forceinline__ void tile_read_scales(const uint8_t* __restrict__ smem, int a_off, int b_off, TileScales<S>& r) {
#pragma unroll
    for (int i = 0; i < S::TM; ++i) r.a[i] = *reinterpret_cast<const uint4*>(smem + a_off + i * 32 * 16);
#pragma unroll
    for (int j = 0; j < S::TN; ++j) r.b[j] = *reinterpret_cast<const uint4*>(smem + b_off + j * 32 * 16);
}
template <int Q>
__device__ __forceinline__ uint32_t dword_of(const uint4& v) {
    return Q == 0 ? v.x : Q == 1 ? v.y : Q == 2 ? v.z : v.w;
}
// the dwords from `by` on first (uniform)
__device__ __forceinline__ uint4 rotate_dwords(uint4 v, int by) {
    if (by & 1) v = make_uint4(v.y, v.z, v.w, v.x);
    if (by & 2) v = make_uint4(v.z, v.w, v.x, v.y);
    return v;
}

// The blocks of four K steps from `first` up to `end` whose format flag is `want`, in ascending order.  flags: one bit per block,
// in LDS; every wave walks them alike.
struct BlockWalk {
    const uint64_t* flags;
    uint64_t word;
    int base, end;
    uint32_t invert;
    __device__ __forceinline__ uint64_t load(int at) const {
        const uint2 v = *reinterpret_cast<const uint2*>(flags + (at >> 6));
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)v.x), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)v.y);
        return ((uint64_t)(hi ^ invert) << 32) | (lo ^ invert);
    }
    __device__ __forceinline__ BlockWalk(const uint8_t* f, int first, int last, bool want)
        : flags(reinterpret_cast<const uint64_t*>(f)), base(first & ~63), end(last), invert(want ? 0u : ~0u) {
        word = load(base) & (~0ull << (first & 63));
    }
    __device__ __forceinline__ int next() {   // `end` behind the last one, and from then on
        while (!word) {
            if (base + 64 >= end) return end;
            base += 64;
            word = load(base);
        }
        const int b = base + __builtin_ctzll(word);
        word &= word - 1;
        return b < end ? b : end;
    }
};

// `count` of them (uniform), zeros behind
__device__ __forceinline__ uint4 first_dwords(uint4 v, int count) { return make_uint4(v.x, count > 1 ? v.y : 0u, count > 2 ? v.z : 0u, 0u); }

template <class S>
struct TileFrags {
    uint4 a[S::TM], b[S::TN * S::kBBlocks];
};
template <class S>
__device__ __forceinline__ void tile_read(const uint8_t* __restrict__ stage, int a_off, int b_off, TileFrags<S>& f) {
#pragma unroll
    for (int i = 0; i < S::TM; ++i) f.a[i] = *reinterpret_cast<const uint4*>(stage + a_off + i * 32 * kRowBytes);
#pragma unroll
    for (int j = 0; j < S::TN; ++j)
#pragma unroll
        for (int q = 0; q < S::kBBlocks; ++q)
            f.b[j * S::kBBlocks + q] = *reinterpret_cast<const uint4*>(stage + b_off + q * S::BN * kRowBytes + j * 32 * kRowBytes);
}
// SWAP: B's rows (n) are the instruction's first operand, so a lane ends up with quads of consecutive n of one m
template <class S, int SUB, bool SWAP, bool ZERO, bool SIX = false>
__device__ __forceinline__ void tile_mfma_row(int i, const TileFrags<S>& f, const uint32_t (&sca)[S::TM], const uint32_t (&scb)[S::TN],
                                              v16f (&acc)[S::TM][S::TN]) {
    {
        const v8i av = v8i{(int)f.a[i].x, (int)f.a[i].y, (int)f.a[i].z, (int)f.a[i].w, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < S::TN; ++j) {
            // eight-bit operand: a lane holds sixteen bytes of either block of 32 indices, low registers first (FP4: a whole block)
            const uint4 b0 = f.b[j * S::kBBlocks], b1 = S::kWideB ? f.b[j * S::kBBlocks + S::kBBlocks - 1] : make_uint4(0u, 0u, 0u, 0u);
            const v8i bv = v8i{(int)b0.x, (int)b0.y, (int)b0.z, (int)b0.w, (int)b1.x, (int)b1.y, (int)b1.z, (int)b1.w};
            constexpr int kFmtB = SIX ? 3 : S::kWideB ? 1 : 4;   // E3M2 (24 of the 32 bytes count), E5M2, E2M1
            v16f cin;
            if constexpr (ZERO) {
#pragma unroll
                for (int e = 0; e < 16; ++e) cin[e] = 0.0f;
            } else {
                cin = acc[i][j];
            }
            if constexpr (SWAP)
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bv, av, cin, kFmtB, 4, SUB, (int)scb[j], SUB, (int)sca[i]);
            else
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, cin, 4, kFmtB, SUB, (int)sca[i], SUB, (int)scb[j]);
        }
    }
}

template <class S, int SUB, bool SWAP, bool ZERO, bool SIX = false>
__device__ __forceinline__ void tile_mfma(const TileFrags<S>& f, const uint32_t (&sca)[S::TM], const uint32_t (&scb)[S::TN],
                                          v16f (&acc)[S::TM][S::TN]) {
#pragma unroll
    for (int i = 0; i < S::TM; ++i) tile_mfma_row<S, SUB, SWAP, ZERO, SIX>(i, f, sca, scb, acc);
}

// ROT: the masked inverse rotation in the epilogue (bf16 results of the product).  A template argument: a plain product that carries
// the rotation's code behind a branch is slower with the same registers (an inference call of 1000 x 1536 x 8192 15.8 us, 15.5
// without; an evaluated 30 M model's pass 1000 and 992).
// Evaluated 30 M model, 4096 tokens: 4096 x 3456 x 640 with SwiGLU and quantizer in its end 16.1 us (256 x 128 tiles 17.7), 12.7 and 12.5 as two
// launches; 4096 x 1920 x 640 with the rotary split 12.3 us, 16.4 as two; a pass of the model 1004 -> 924.  What bounds them: the 1400
// vector instructions of a group's quantizer, three waves to a SIMD, and a second round of few tiles.
// AFTER: what becomes of a plain bf16 result in an evaluated model, instead of being stored (TileAfter): nothing else, the SwiGLU of its two
// halves quantized for the next layer, or its split into q, k and v with the rotary embedding.
enum TileEnd : int { END_STORE = 0, END_SWIGLU = 1, END_ROPE = 2 };
template <class S, typename OutT, bool ROT, int AFTER = END_STORE>
__device__ __forceinline__ void tile_run(const TileProduct& g, int t, uint32_t* smem, uint32_t smem_base, [[maybe_unused]] const TileAfter& after = TileAfter{}) {
    static_assert(AFTER == END_STORE || (sizeof(OutT) == 2 && !ROT && !S::kWideB), "ends of plain bf16 products");
    constexpr bool SWAP = sizeof(OutT) == 2;
    uint8_t* smem_bytes = reinterpret_cast<uint8_t*>(smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / S::kWavesN, wn = wave % S::kWavesN;
    const int lrow = lane & 31, half = lane >> 5;
    const int M = g.M, N = g.N, K = g.K;
    // SwiGLU: half of a tile's columns are of the one half of B's rows, half the same columns of the other; with the next layer's padding
    const int hidden = N / 2, hidden_groups = hidden / 32, hidden_padded = (hidden_groups + 3) & ~3;
    const int tiles_m = (M + S::BM - 1) / S::BM, tiles_n = AFTER == END_SWIGLU ? (hidden_padded * 64 + S::BN - 1) / S::BN : (N + S::BN - 1) / S::BN;
    const int code_pitch = K / 2, groups = K / 32;
    // a work item is (tile, K range): range r covers steps [r * all / splits, (r + 1) * all / splits) and, with splits > 1 (fp32
    // instantiation only), stores its partial sums, unscaled, into slab r of c = [splits][M][N]
    const int tiles = tiles_m * tiles_n, item = xcd_run(t, tiles * g.splits), range = item / tiles;
    const int nk_all = (K + kBK - 1) / kBK;
    const int k_first = S::kMixed ? 0 : range * nk_all / g.splits, nk = (range + 1) * nk_all / g.splits - k_first;
    const int half_step = (K % kBK) && range == g.splits - 1 ? nk - 1 : -1;  // the K step that covers only 64 indices (K % 128 == 64), or none
    int tm, tn;
    tile_of_run<(S::BM >= 256 ? 4 : 8)>(item - range * tiles, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * S::BM, n0 = tn * S::BN;
    const int h0 = tn * (S::BN / 2);
    // the packed operand's place of group gh of a row, in 16-byte pieces
    const auto packed_slot = [&](int row, int gh) { return (int64_t)(row >> 4) * 16 * hidden_padded + ((gh >> 2) * 64 + (row & 15) * 4 + (gh & 3)); };
    if constexpr (AFTER == END_SWIGLU)
        if (h0 >= hidden) {   // a tile of padding: zero codes and scales
            for (int u = tid; u < S::BM * (S::BN / 64); u += S::kThreads) {
                const int row = m0 + u / (S::BN / 64), gh = h0 / 32 + u % (S::BN / 64);
                if (row >= M || gh >= hidden_padded) continue;
                reinterpret_cast<uint4*>(g.c)[packed_slot(row, gh)] = make_uint4(0u, 0u, 0u, 0u);
                after.scales[(int64_t)row * hidden_padded + gh] = 0;
            }
            return;
        }
    const auto source_of = [&](int r) {   // B's row behind column r of the tile
        const int h = h0 + r % (S::BN / 2) < hidden ? h0 + r % (S::BN / 2) : hidden - 1;
        return r < S::BN / 2 ? h : hidden + h;
    };

    const int swz = (lrow >> 2) & 3;
    const int a_off0 = (wm * S::WM + lrow) * kRowBytes + (((2 * half) ^ swz) * 16);
    const int a_off1 = (wm * S::WM + lrow) * kRowBytes + (((2 * half + 1) ^ swz) * 16);
    // the 16-byte pieces of B's row for the two halves of a K step: block 2 * half + sub of 32 codes; with eight-bit values bytes
    // 16 * half of block sub in the first 64 indices and of block 2 + sub in the second
    const int b_off0 = S::kBOff + (wn * S::WN + lrow) * kRowBytes + (((S::kWideB ? half : 2 * half) ^ swz) * 16);
    const int b_off1 = S::kBOff + (wn * S::WN + lrow) * kRowBytes + (((S::kWideB ? 2 + half : 2 * half + 1) ^ swz) * 16);
    // scales in LDS: A dword p holds row (p / (32 TM)) * WM + (p % TM) * 32 + (p / TM) % 32, so one read fetches the scale
    // dwords of a lane's TM blocks; B likewise with TN and WN
    // (BLOCKS: 16 bytes per row, in the rows' order)
    const int a_sc_off = S::kSAOff + (S::kBlocks ? (wm * S::WM + lrow) * 16 : (wm * 32 + lrow) * (4 * S::TM));
    const int b_sc_off = S::kSBOff + (S::kBlocks ? (wn * S::WN + lrow) * 16 : (wn * 32 + lrow) * (4 * S::TN));
    const int sh = 16 * half;

    TilePlan<S> plan;
    {
        const int prow = lane >> 2;
        const int pcv = (lane & 3) ^ ((prow >> 2) & 3);
        const int64_t row16 = (int64_t)16 * code_pitch;
        const int last_a = (g.a_tiled ? (M + 15) & ~15 : M) - 1 - m0, last_b = (g.b_tiled ? (N + 15) & ~15 : N) - 1 - n0;
        // 16 rows are row16 bytes in either layout
        const uint32_t row_a = g.a_tiled ? 64u : (uint32_t)code_pitch, row_b = g.b_tiled ? 64u : (uint32_t)code_pitch;
        const auto row_off = [&](int r, uint32_t row_bytes) { return (uint32_t)(r >> 4) * (uint32_t)row16 + (uint32_t)(r & 15) * row_bytes + pcv * 16; };
        plan.kstep_a = g.a_tiled ? 1024 : kRowBytes;
        plan.kstep_b = g.b_tiled ? 1024 * S::kBBlocks : kRowBytes;
        plan.a = g.a_codes + (int64_t)m0 * code_pitch + (int64_t)k_first * plan.kstep_a;   // m0, n0 are multiples of 16: the same
        plan.b = g.b_codes + (AFTER == END_SWIGLU ? 0 : (int64_t)n0 * code_pitch * S::kBBlocks) + (int64_t)k_first * plan.kstep_b;   //   expression in both layouts
#pragma unroll
        for (int j = 0; j < S::kALoads; ++j) {
            const int r = (wave * S::kALoads + j) * 16 + prow;
            plan.voff_a[j] = row_off(r < last_a ? r : last_a, row_a);
        }
#pragma unroll
        for (int j = 0; j < S::kBLoads; ++j) {
            const int u = wave * S::kBLoads + j, r = (u % (S::BN / 16)) * 16 + prow;   // eight-bit B: every column's first 64 indices, then the second
            const int rr = r < last_b ? r : last_b;
            if constexpr (S::kWideB)
                plan.voff_b[j] = (uint32_t)((rr >> 4) * 2 * row16) + (uint32_t)((u / (S::BN / 16)) * 1024 + (rr & 15) * 64 + pcv * 16);
            else
                plan.voff_b[j] = row_off(AFTER == END_SWIGLU ? source_of(r) : rr, row_b);
        }
        plan.half_back = (uint32_t)(pcv & 2) * 16u;
        plan.lds_a = (uint32_t)__builtin_amdgcn_readfirstlane((int)(smem_base + wave * S::kALoads * 1024));
        plan.lds_b = (uint32_t)__builtin_amdgcn_readfirstlane((int)(smem_base + S::kBOff + wave * S::kBLoads * 1024));
#pragma unroll
        for (int u = 0; u < S::kSLoads; ++u) {
            // unit of 64 scale dwords this wave requests; a wave without one of its own repeats another's (same bytes to the
            // same place), which keeps every wave's count of outstanding requests the same
            const int unit = (wave + u * S::kWaves) % S::kUnits;
            const bool is_a = unit < S::kAUnits;
            const int p = (is_a ? unit : unit - S::kAUnits) * 64 + lane;
            const int ra = S::kBlocks ? p : (p / (32 * S::TM)) * S::WM + (p % S::TM) * 32 + (p / S::TM) % 32;
            const int rb = S::kBlocks ? p : (p / (32 * S::TN)) * S::WN + (p % S::TN) * 32 + (p / S::TN) % 32;
            const int la = M - 1 - m0, lb = N - 1 - n0;
            const int r = is_a ? (ra < la ? ra : la) : AFTER == END_SWIGLU ? source_of(rb) : (rb < lb ? rb : lb);
            plan.s[u] = (is_a ? g.a_scales + (int64_t)m0 * groups : g.b_scales + (AFTER == END_SWIGLU ? 0 : (int64_t)n0 * groups)) + k_first * 4;
            plan.voff_s[u] = (uint32_t)(r * groups);
            plan.lds_s[u] = (uint32_t)__builtin_amdgcn_readfirstlane((int)(smem_base + S::kSAOff + unit * S::kUnitBytes));
        }
    }
    // The rotation's mask words of the tile, [BM][BN / 32] in LDS: with room beside the ring they are requested ahead of
    // the operands, otherwise into the ring's free end once the K loop is done.
    const auto issue_mask = [&](uint32_t at) {
        const int64_t pitch = N / 8;   // N is a multiple of 32 with a mask: whole words
        const uint8_t* base = g.mask + (int64_t)m0 * pitch;
#pragma unroll
        for (int u = 0; u < S::kMLoads; ++u) {
            const int unit = (wave + u * S::kWaves) % S::kMUnits;
            const int p = unit * 64 + lane, r = p / (S::BN / 32);
            const int col = n0 / 32 + p % (S::BN / 32);
            const int rr = r < M - 1 - m0 ? r : M - 1 - m0, cc = col < N / 32 ? col : N / 32 - 1;
            load_lds_b32_s(base, (uint32_t)(rr * (int)pitch + cc * 4),
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)(smem_base + at + unit * 256)));
        }
    };
    if constexpr (ROT && S::kMaskEarly) issue_mask(S::kMaskOff);

    const auto issue = [&](int stage, int ks) { tile_issue<S>(plan, stage, ks, ks == half_step); };
    const auto live_until = [&](int ks) { return ks < nk ? ~0u : 0u; };
    // the scale dwords of a half step arrive two bytes early (see tile_issue).  Without a branch: a K step is one basic block.
    const auto settle_scales = [&](uint32_t (&a)[S::TM], uint32_t (&b)[S::TN], int ks) {
        const uint32_t down = ks == half_step ? 16u : 0u;
#pragma unroll
        for (int i = 0; i < S::TM; ++i) a[i] >>= down;
#pragma unroll
        for (int j = 0; j < S::TN; ++j) b[j] >>= down;
    };
    TileFrags<S> f0, f1;
    v16f acc[S::TM][S::TN];
    int stage = 0;
    if constexpr (S::kMixed) {
        // B's blocks of four K steps in six bits, then those in eight: two passes of the same loop, each over its blocks, so that a
        // block costs what its format does (all in eight bits: as without this; every second one: half way).  The short last block
        // of a K that is no multiple of four steps is filled up with muted ones: a tail of its own, as below, makes the compiler
        // keep the accumulators in memory.
        const int blocks_all = (nk_all + 3) / 4, b_end = (range + 1) * blocks_all / g.splits;
        const uint8_t* flags = g.b_wide + (int64_t)(n0 / kWideStrip) * blocks_all;
        for (int base = wave * 64; base < blocks_all; base += S::kThreads) {
            const uint64_t bits = __builtin_amdgcn_ballot_w64(base + lane < blocks_all && flags[base + lane < blocks_all ? base + lane : 0] != 0);
            if (lane == 0) *reinterpret_cast<uint2*>(smem_bytes + S::kFlagOff + base / 8) = make_uint2((uint32_t)bits, (uint32_t)(bits >> 32));
        }
#pragma unroll
        for (int i = 0; i < S::TM; ++i)
#pragma unroll
            for (int j = 0; j < S::TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
        __syncthreads();
        const auto phase = [&](auto six_tag) {
            constexpr bool SIX = decltype(six_tag)::value;
            constexpr int kB = SIX ? S::kBLoads6 : S::kBLoads, kLoads = S::kALoads + kB;
            BlockWalk walk(smem_bytes + S::kFlagOff, range * blocks_all / g.splits, b_end, !SIX);
            int block = walk.next();
            if (block == b_end) return;
            uint32_t voff_b[kB], lds_b[kB];
#pragma unroll
            for (int j = 0; j < kB; ++j) {
                // six bits: every column's 16 bytes of a block of 32 indices, then, by 32 columns, its 8 bytes
                const int u = SIX ? (wave * kB + j) % S::kUnits6 : wave * kB + j, pair = u - S::BN / 16;
                if (SIX && pair >= 0) {
                    const int last_pair = (N - 1 - n0) >> 5;
                    voff_b[j] = (uint32_t)(pair < last_pair ? pair : last_pair) * (uint32_t)(32 * K) + 1024u + lane * 16;
                } else {
                    const int r = (u % (S::BN / 16)) * 16 + (lane >> 2), rr = r < N - 1 - n0 ? r : N - 1 - n0;
                    voff_b[j] = (uint32_t)(rr >> 4) * (uint32_t)(16 * K) + (uint32_t)((u / (S::BN / 16)) * 1024 + (rr & 15) * 64 + ((lane & 3) ^ ((lane >> 4) & 3)) * 16);
                }
                lds_b[j] = (uint32_t)__builtin_amdgcn_readfirstlane((int)(smem_base + S::kBOff + u * 1024));
            }
            const auto issue_one = [&](int slot, int ks, int l) {
                ks = ks < nk_all ? ks : nk_all - 1;
                const uint32_t off = (uint32_t)slot * S::kStageBytes;
                if (l < S::kALoads) load_lds_b128_s(plan.a + (int64_t)ks * plan.kstep_a, plan.voff_a[l], plan.lds_a + off + l * 1024);
                else load_lds_b128_s(plan.b + (int64_t)ks * plan.kstep_b, voff_b[l - S::kALoads], lds_b[l - S::kALoads] + off);
            };
            const auto issue = [&](int slot, int ks) {
#pragma unroll
                for (int l = 0; l < kLoads; ++l) issue_one(slot, ks, l);
            };
            const auto scales_at = [&](int b) { return 4 * b + 4 <= nk_all ? 4 * b : nk_all - 4; };   // the last block: its row's final 16 bytes
            const auto read_row = [&](const uint8_t* slot, int sub, TileFrags<S>& f, int i) {
                f.a[i] = *reinterpret_cast<const uint4*>(slot + (sub ? a_off1 : a_off0) + i * 32 * kRowBytes);
                if (const int j = i; j < S::TN) {
                    if constexpr (SIX) {
                        const int piece = 2 * half + sub;
                        f.b[2 * j] = *reinterpret_cast<const uint4*>(slot + S::kBOff + (wn * S::WN + j * 32 + lrow) * kRowBytes + ((piece ^ swz) * 16));
                        const uint2 v = *reinterpret_cast<const uint2*>(slot + S::kBOff + S::BN * kRowBytes + (wn * (S::WN / 32) + j) * 1024 + piece * 256 + lrow * 8);
                        f.b[2 * j + 1] = make_uint4(v.x, v.y, 0u, 0u);
                    } else {
                        f.b[2 * j] = *reinterpret_cast<const uint4*>(slot + (sub ? b_off1 : b_off0) + j * 32 * kRowBytes);
                        f.b[2 * j + 1] = *reinterpret_cast<const uint4*>(slot + (sub ? b_off1 : b_off0) + S::BN * kRowBytes + j * 32 * kRowBytes);
                    }
                }
            };
            const auto read = [&](const uint8_t* slot, int sub, TileFrags<S>& f) {
#pragma unroll
                for (int i = 0; i < S::TM; ++i) read_row(slot, sub, f, i);
            };
            int stage = 0;
            tile_issue_scales<S>(plan, scales_at(block));
#pragma unroll
            for (int s = 0; s < S::STAGES; ++s) issue(s, 4 * block + s);
            __builtin_amdgcn_s_waitcnt(vmcnt_imm((S::STAGES - 1) * kLoads));
            __syncthreads();
            TileScales<S> sc;
            tile_read_scales<S>(smem_bytes, a_sc_off, b_sc_off, sc);
            read(smem_bytes, 0, f0);
            int next = block;
            // one K step, as below; the requests of a block's last steps are the first ones of the block that follows it here.
            // Requests, reads and products dealt out by 32 rows, where they otherwise stand between the barrier and the first
            // product: 59.2 -> 58.3 us at 4096^3 (with the rotation as it was then, see rotate_rows).
            auto step = [&](auto q_tag) {
                constexpr int Q = decltype(q_tag)::value;
                const int nstage = stage == S::STAGES - 1 ? 0 : stage + 1;
                const uint8_t* cur = smem_bytes + stage * S::kStageBytes;
                const uint8_t* nxt = smem_bytes + nstage * S::kStageBytes;
                uint32_t sca[S::TM], scb[S::TN];
#pragma unroll
                for (int i = 0; i < S::TM; ++i) sca[i] = __builtin_amdgcn_ubfe(dword_of<Q>(sc.a[i]), (uint32_t)sh, 16u);
#pragma unroll
                for (int j = 0; j < S::TN; ++j) scb[j] = __builtin_amdgcn_ubfe(dword_of<Q>(sc.b[j]), (uint32_t)sh, 16u);
                read(cur, 1, f1);
                tile_mfma<S, 0, SWAP, false, SIX>(f0, sca, scb, acc);
                if constexpr (S::TM * S::TN >= S::TM + S::TN) { QM_SCHED_PAIR(0x100, S::TM + S::TN * 2) }
                __builtin_amdgcn_sched_barrier(0);
                constexpr int kPending = (S::STAGES - 2) * kLoads + (Q >= 1 && Q <= S::STAGES - 1 ? S::kSLoads : 0);
                __builtin_amdgcn_s_waitcnt(vmcnt_imm(Q == 3 && kPending > 2 * kLoads ? 2 * kLoads : kPending));
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
                const int ks = Q + S::STAGES < 4 ? 4 * block + Q + S::STAGES : 4 * next + Q + S::STAGES - 4;
                if constexpr (Q == 3) tile_read_scales<S>(smem_bytes, a_sc_off, b_sc_off, sc);
#pragma unroll
                for (int i = 0; i < S::TM; ++i) {   // a request or two, the reads, the products of every 32 rows
#pragma unroll
                    for (int l = i * kLoads / S::TM; l < (i + 1) * kLoads / S::TM; ++l) issue_one(stage, ks, l);
                    if (Q == 0 && i == S::TM - 1) tile_issue_scales<S>(plan, scales_at(next));
                    read_row(nxt, 0, f0, i);
                    tile_mfma_row<S, 1, SWAP, false, SIX>(i, f1, sca, scb, acc);
                    __builtin_amdgcn_sched_barrier(0);
                }
                stage = nstage;
            };
            for (bool more = true; more;) {
                // K no multiple of four steps: the last block's dwords are the last ones of its 16 bytes, and the steps that it
                // lacks repeat its last one with scales of 2^-127 on both sides, whose products vanish
                if (const int left = nk_all - 4 * block; left < 4) {
#pragma unroll
                    for (int i = 0; i < S::TM; ++i) sc.a[i] = first_dwords(rotate_dwords(sc.a[i], 4 - left), left);
#pragma unroll
                    for (int j = 0; j < S::TN; ++j) sc.b[j] = first_dwords(rotate_dwords(sc.b[j], 4 - left), left);
                }
                next = walk.next();
                more = next < b_end;
                next = more ? next : block;
                step(std::integral_constant<int, 0>{});
                step(std::integral_constant<int, 1>{});
                step(std::integral_constant<int, 2>{});
                step(std::integral_constant<int, 3>{});
                block = next;
            }
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
            __syncthreads();
        };
        phase(std::true_type{});
        phase(std::false_type{});
    } else if constexpr (S::kBlocks) {
        // blocks of four K steps; the last block of an nk that is no multiple of four requests the row's final 16 bytes, whose
        // first dwords the block before has used
        const auto block_at = [&](int ks) { return ks + 4 <= nk ? ks : nk - 4; };
        tile_issue_scales<S>(plan, 0);
#pragma unroll
        for (int s = 0; s < S::STAGES; ++s) tile_issue<S>(plan, s, s < nk ? s : nk - 1, false, live_until(s));   // whole steps: K is a multiple of 128
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((S::STAGES - 1) * S::kLoads));  // the scales and step 0 are in; later ones may be pending
        __syncthreads();
        TileScales<S> sc;
        tile_read_scales<S>(smem_bytes, a_sc_off, b_sc_off, sc);
        tile_read<S>(smem_bytes, a_off0, b_off0, f0);
        // one K step, dword Q of its block's scales: `stage` is the ring slot it consumes and then refills with step s + STAGES
        auto step = [&](auto first_tag, auto q_tag, int s) {
            constexpr bool FIRST = decltype(first_tag)::value;
            constexpr int Q = decltype(q_tag)::value;
            const int nstage = stage == S::STAGES - 1 ? 0 : stage + 1;
            const uint8_t* cur = smem_bytes + stage * S::kStageBytes;
            const uint8_t* nxt = smem_bytes + nstage * S::kStageBytes;
            uint32_t sca[S::TM], scb[S::TN];
#pragma unroll
            for (int i = 0; i < S::TM; ++i) sca[i] = __builtin_amdgcn_ubfe(dword_of<Q>(sc.a[i]), (uint32_t)sh, 16u);
#pragma unroll
            for (int j = 0; j < S::TN; ++j) scb[j] = __builtin_amdgcn_ubfe(dword_of<Q>(sc.b[j]), (uint32_t)sh, 16u);
            tile_read<S>(cur, a_off1, b_off1, f1);
            tile_mfma<S, 0, SWAP, FIRST>(f0, sca, scb, acc);
            if constexpr (S::TM * S::TN >= S::TM + S::TN) { QM_SCHED_PAIR(0x100, S::TM + S::TN * S::kBBlocks) }
            __builtin_amdgcn_sched_barrier(0);
            // younger than the requests of step s + 1: those of the STAGES - 2 steps after it, and the scales requested in this
            // block's first step where that is one of them; the next block's scales, which the block's last step reads, are younger
            // than all but the requests of two steps
            constexpr int kPending = (S::STAGES - 2) * S::kLoads + (Q >= 1 && Q <= S::STAGES - 1 ? S::kSLoads : 0);
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(Q == 3 && kPending > 2 * S::kLoads ? 2 * S::kLoads : kPending));
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
            // past the end: a request nobody reads
            tile_issue<S>(plan, stage, s + S::STAGES < nk ? s + S::STAGES : nk - 1, false, live_until(s + S::STAGES));
            if constexpr (Q == 0) tile_issue_scales<S>(plan, block_at(s + 4), live_until(s + 4));   // every wave has taken this block's scales
            if constexpr (Q == 3) tile_read_scales<S>(smem_bytes, a_sc_off, b_sc_off, sc);
            tile_read<S>(nxt, a_off0, b_off0, f0);
            tile_mfma<S, 1, SWAP, false>(f1, sca, scb, acc);
            if constexpr (S::TM * S::TN >= S::TM + S::TN) { QM_SCHED_PAIR(0x100, S::TM + S::TN * S::kBBlocks) }
            __builtin_amdgcn_sched_barrier(0);
            stage = nstage;
        };
        using Q0 = std::integral_constant<int, 0>;
        using Q1 = std::integral_constant<int, 1>;
        using Q2 = std::integral_constant<int, 2>;
        using Q3 = std::integral_constant<int, 3>;
        // (four bodies with a way out behind each, instead of a first block, a loop and a tail, are slower: 42 us for 40 at
        // 4608 x 1536 x 8192, 83 for 71 with the eight-bit B of 4096^3)
        const auto rest_of_block = [&](int ks) {
            step(std::false_type{}, Q1{}, ks + 1);
            step(std::false_type{}, Q2{}, ks + 2);
            step(std::false_type{}, Q3{}, ks + 3);
        };
        step(std::true_type{}, Q0{}, 0);
        rest_of_block(0);
        int ks = 4;
        for (; ks + 4 <= nk; ks += 4) {
            step(std::false_type{}, Q0{}, ks);
            rest_of_block(ks);
        }
        if (const int left = nk - ks; left > 0) {   // the short block's dwords are the last ones of its 16 bytes
#pragma unroll
            for (int i = 0; i < S::TM; ++i) sc.a[i] = rotate_dwords(sc.a[i], 4 - left);
#pragma unroll
            for (int j = 0; j < S::TN; ++j) sc.b[j] = rotate_dwords(sc.b[j], 4 - left);
            step(std::false_type{}, Q0{}, ks);
            if (left > 1) step(std::false_type{}, Q1{}, ks + 1);
            if (left > 2) step(std::false_type{}, Q2{}, ks + 2);
        }
    } else {
#pragma unroll
        for (int s = 0; s < S::STAGES; ++s) issue(s, s < nk ? s : nk - 1);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((S::STAGES - 1) * S::kLoads));  // step 0 is in; later ones may be pending
        __syncthreads();
        uint32_t sa[S::TM], sb[S::TN];
        read_dwords<S::TM>(smem_bytes + a_sc_off, sa);
        read_dwords<S::TN>(smem_bytes + b_sc_off, sb);
        settle_scales(sa, sb, 0);
        tile_read<S>(smem_bytes, a_off0, b_off0, f0);

        // one K step: `stage` is the ring slot it consumes and then refills with step s + STAGES
        auto step = [&](auto first_tag, int s) {
            constexpr bool FIRST = decltype(first_tag)::value;
            const int nstage = stage == S::STAGES - 1 ? 0 : stage + 1;
            const uint8_t* cur = smem_bytes + stage * S::kStageBytes;
            const uint8_t* nxt = smem_bytes + nstage * S::kStageBytes;
            uint32_t sca[S::TM], scb[S::TN];
#pragma unroll
            for (int i = 0; i < S::TM; ++i) sca[i] = __builtin_amdgcn_ubfe(sa[i], (uint32_t)sh, 16u);
#pragma unroll
            for (int j = 0; j < S::TN; ++j) scb[j] = __builtin_amdgcn_ubfe(sb[j], (uint32_t)sh, 16u);
            tile_read<S>(cur, a_off1, b_off1, f1);
            tile_mfma<S, 0, SWAP, FIRST>(f0, sca, scb, acc);
            if constexpr (S::TM * S::TN >= S::TM + S::TN) { QM_SCHED_PAIR(0x100, S::TM + S::TN * S::kBBlocks) }
            __builtin_amdgcn_sched_barrier(0);
            // younger than the requests of step s + 1: those of the STAGES - 2 steps after it
            __builtin_amdgcn_s_waitcnt(vmcnt_imm((S::STAGES - 2) * S::kLoads));
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
            // past the end: a repeat nobody reads keeps the counts of outstanding requests uniform
            issue(stage, s + S::STAGES < nk ? s + S::STAGES : nk - 1);
            read_dwords<S::TM>(nxt + a_sc_off, sa);
            read_dwords<S::TN>(nxt + b_sc_off, sb);
            settle_scales(sa, sb, s + 1);
            tile_read<S>(nxt, a_off0, b_off0, f0);
            tile_mfma<S, 1, SWAP, false>(f1, sca, scb, acc);
            if constexpr (S::TM * S::TN >= S::TM + S::TN) { QM_SCHED_PAIR(0x100, S::TM + S::TN * S::kBBlocks) }
            __builtin_amdgcn_sched_barrier(0);
            stage = nstage;
        };
        step(std::true_type{}, 0);
        for (int ks = 1; ks < nk; ++ks) step(std::false_type{}, ks);
    }
    // every request has landed and every wave has read its last fragments: the ring becomes the staging area
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __syncthreads();
    const float alpha = g.splits > 1 ? 1.0f : g.alpha;
    if constexpr (ROT && !S::kMaskEarly) issue_mask(S::kMaskOff);
    if constexpr (SWAP) {
#pragma unroll
        for (int i = 0; i < S::TM; ++i)
#pragma unroll
            for (int j = 0; j < S::TN; ++j)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const v16f& v = acc[i][j];
                    const v2bf p0 = __builtin_convertvector(v2f{v[4 * b] * alpha, v[4 * b + 1] * alpha}, v2bf);
                    const v2bf p1 = __builtin_convertvector(v2f{v[4 * b + 2] * alpha, v[4 * b + 3] * alpha}, v2bf);
                    *reinterpret_cast<uint2*>(smem_bytes + (wm * S::WM + i * 32 + lrow) * S::kPitch + (wn * S::WN + j * 32 + 8 * b + 4 * half) * 2) =
                        make_uint2(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1));
                }
        if constexpr (ROT && !S::kMaskEarly) __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        __syncthreads();
        // an opaque copy: what is worked out from it (the rotation's signs, addresses) otherwise holds 16 to 38 registers from ahead of
        // the loop over tiles on, through every K step, and up to 200 bytes a lane of scratch (an error-only step of 4096^3 187 us, now 183)
        int id = tid;
        if constexpr (ROT) asm volatile("" : "+v"(id));
        const int chunk = id % S::kChunks, rsub = id / S::kChunks;
        const int out_col = n0 + chunk * 8;
        typedef uint32_t u4v __attribute__((ext_vector_type(4)));
        typedef float f4v __attribute__((ext_vector_type(4)));
        const bool col_ok = out_col < N;   // N is a multiple of 8
        if constexpr (AFTER == END_SWIGLU) {
            // A lane per row and group: the arithmetic of the producer (SwiGluProducer) and the quantizer on the bf16 values that would
            // have been stored, the same bits; no clip mask, which only a backward pass reads.
            constexpr int kSide = S::BN / 64;   // groups of the next operand per row of the tile
#pragma unroll 1
            for (int u = id; u < S::BM * kSide; u += S::kThreads) {
                const int line = u / kSide, row = m0 + line, side = u % kSide, gh = h0 / 32 + side;
                const auto read_group = [&](int at, float (&v)[32]) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint4 raw = *reinterpret_cast<const uint4*>(smem_bytes + line * S::kPitch + at + q * 16);
                        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            v[8 * q + 2 * e] = u2f(w[e] << 16);
                            v[8 * q + 2 * e + 1] = u2f(w[e] & 0xffff0000u);
                        }
                    }
                };
                float v[32], gate[32];
                read_group(side * 64, v);
                read_group(S::BN + side * 64, gate);
                swiglu_group_bf16(v, gate);
                rotate_group(v, after.c, after.sign_word);
                GroupCodes o;
                quantize_group_regs<QUEST_RTN, false>(v, 0, 0, o);
                if (row >= M || gh >= hidden_padded) continue;
                const bool real = gh < hidden_groups;
                reinterpret_cast<uint4*>(g.c)[packed_slot(row, gh)] = real ? make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]) : make_uint4(0u, 0u, 0u, 0u);
                after.scales[(int64_t)row * hidden_padded + gh] = real ? (uint8_t)o.scale_byte : 0;
            }
        } else if constexpr (AFTER == END_ROPE) {
            // (q, k, v) by thirds of the columns, pairs of q and k rotated in fp32: the arithmetic of rope_qkv_kernel on the bf16 values that
            // would have been stored, the same bits
            const int part = out_col / after.width, c = out_col - part * after.width, pair = (c % after.head_dim) >> 1;
            uint16_t* dst = static_cast<uint16_t*>(part == 0 ? after.q : part == 1 ? after.k : after.v);
            constexpr int kAtOnce = S::kPasses < 4 ? S::kPasses : 4;   // passes whose table entries are on their way together
            int pos = (m0 + rsub) % after.seq_len;
#pragma unroll 1
            for (int r0 = 0; r0 < S::kPasses; r0 += kAtOnce) {
                float4 t[kAtOnce][2];
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i) {
                    if (part < 2) {   // rows past the end have positions, too
                        const float4* cs = reinterpret_cast<const float4*>(after.table + ((int64_t)pos * (after.head_dim / 2) + pair) * 2);
                        t[i][0] = cs[0];
                        t[i][1] = cs[1];
                    }
                    for (pos += S::kRowsPerPass; pos >= after.seq_len;) pos -= after.seq_len;
                }
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i) {
                    const int line = (r0 + i) * S::kRowsPerPass + rsub, row = m0 + line;
                    uint4 v = *reinterpret_cast<const uint4*>(smem_bytes + line * S::kPitch + chunk * 16);
                    const auto turn = [](uint32_t w, float co, float si) {
                        const float a = u2f(w << 16), b = u2f(w & 0xffff0000u);
                        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{a * co - b * si, a * si + b * co}, v2bf));
                    };
                    if (part < 2)
                        v = make_uint4(turn(v.x, t[i][0].x, t[i][0].y), turn(v.y, t[i][0].z, t[i][0].w), turn(v.z, t[i][1].x, t[i][1].y), turn(v.w, t[i][1].z, t[i][1].w));
                    if (col_ok && row < M) *reinterpret_cast<uint4*>(dst + (int64_t)row * after.width + c) = v;
                }
            }
        } else if constexpr (!ROT) {
            uint16_t* out = reinterpret_cast<uint16_t*>(g.c) + (int64_t)(m0 + rsub) * N + out_col;
#pragma unroll
            for (int r = 0; r < S::kPasses; ++r) {
                const uint4 v = *reinterpret_cast<const uint4*>(smem_bytes + (r * S::kRowsPerPass + rsub) * S::kPitch + chunk * 16);
                if (col_ok && m0 + r * S::kRowsPerPass + rsub < M)
                    __builtin_nontemporal_store(u4v{v.x, v.y, v.z, v.w}, reinterpret_cast<u4v*>(out + (int64_t)r * S::kRowsPerPass * N));
            }
        } else {
            // A loop per block size and type, not unrolled: a tile runs this code once or twice per launch, and what bounds it then is
            // fetching instructions.  Unrolled with the choice of the block size inside, 256 x 256 tiles took 8 us longer
            // (4096^3, 59.8 -> 51.8), 128 x 128 ones 2 to 3 (8192 x 2048 x 2048, 46.9 -> 43.2); unrolled twice is no faster.
            const auto rotate_rows = [&](auto hd_tag, auto f32_tag) {
                constexpr int HD = decltype(hd_tag)::value;
                if constexpr (S::BN >= HD) {
#pragma unroll 1
                    for (int r = 0; r < S::kPasses; ++r) {
                        const int line = r * S::kRowsPerPass + rsub, row = m0 + line;
                        const uint4 raw = *reinterpret_cast<const uint4*>(smem_bytes + line * S::kPitch + chunk * 16);
                        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
                        float v[8];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            v[2 * i] = u2f(w[i] << 16);
                            v[2 * i + 1] = u2f(w[i] & 0xffff0000u);
                        }
                        const uint32_t kb = smem_bytes[S::kMaskOff + line * (S::BN / 8) + chunk];
                        // whole Hadamard blocks lie in neighbouring lanes (N is a multiple of the block); lanes past N work along
                        octet_inverse_rotation<HD>(v, kb, chunk & (HD / 8 - 1), g.signs);
                        uint32_t o[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{v[2 * i] * g.rot_c, v[2 * i + 1] * g.rot_c}, v2bf));
                        if constexpr (!decltype(f32_tag)::value) {
                            if (col_ok && row < M)
                                __builtin_nontemporal_store(u4v{o[0], o[1], o[2], o[3]}, reinterpret_cast<u4v*>(reinterpret_cast<uint16_t*>(g.c) + (int64_t)row * N + out_col));
                        } else {
                            // The bf16-rounded result, widened.  A lane's 32 bytes would be every other 16 bytes of two stores, so the
                            // values go back to where they were and the wave stores its rows four values a lane, whole lines: a step
                            // with 8192 x 6656 weights and 448 tokens takes 193 us, 255 with half lines as non-temporal stores, 207 as
                            // others; 4096 x 11008 and 2048 tokens 293, 329 and 306.
                            *reinterpret_cast<uint4*>(smem_bytes + line * S::kPitch + chunk * 16) = make_uint4(o[0], o[1], o[2], o[3]);
                            __builtin_amdgcn_wave_barrier();
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                const int at = h * 256 + (id & 63) * 4, col = at % S::BN, wline = r * S::kRowsPerPass + wave * (64 / S::kChunks) + at / S::BN;
                                const uint2 q = *reinterpret_cast<const uint2*>(smem_bytes + wline * S::kPitch + col * 2);
                                if (n0 + col < N && m0 + wline < M)
                                    __builtin_nontemporal_store(f4v{u2f(q.x << 16), u2f(q.x & 0xffff0000u), u2f(q.y << 16), u2f(q.y & 0xffff0000u)},
                                                                reinterpret_cast<f4v*>(reinterpret_cast<float*>(g.c) + (int64_t)(m0 + wline) * N + n0 + col));
                            }
                        }
                    }
                }
            };
            const auto rotate = [&](auto hd_tag) { g.out_f32 ? rotate_rows(hd_tag, std::true_type{}) : rotate_rows(hd_tag, std::false_type{}); };
            if (g.hd == 32) rotate(std::integral_constant<int, 32>{});
            else if (g.hd == 64) rotate(std::integral_constant<int, 64>{});
            else rotate(std::integral_constant<int, 128>{});
        }
    } else {
        float* c = reinterpret_cast<float*>(g.c) + (int64_t)range * M * N;
#pragma unroll
        for (int i = 0; i < S::TM; ++i)
#pragma unroll
            for (int j = 0; j < S::TN; ++j) {
                const int col = n0 + wn * S::WN + j * 32 + lrow;
                if (col >= N) continue;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int row = m0 + wm * S::WM + i * 32 + 8 * (e / 4) + 4 * half + (e & 3);
                    if (row < M) c[(int64_t)row * N + col] = acc[i][j][e] * alpha;
                }
            }
    }
    __syncthreads();  // the staging area is the next tile's ring
}

template <class S, typename OutT, bool ROT>
__device__ __forceinline__ void run_tiles(const TileProduct& g, int tiles) {   // persistent over the tiles
    extern __shared__ uint32_t smem[];
    const uint32_t smem_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)smem;
    for (int t = (int)blockIdx.x; t < tiles; t += (int)gridDim.x) tile_run<S, OutT, ROT>(g, t, smem, smem_base);
}
template <class S, typename OutT, bool ROT>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu((S::OCC * S::kWaves + 3) / 4))) void gemm_mxfp4_tn_tile_kernel(
    TileProduct g, int tiles) {
    run_tiles<S, OutT, ROT>(g, tiles);
}
// the same with an eight-bit B
template <class S, typename OutT, bool ROT>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu((S::OCC * S::kWaves + 3) / 4))) void gemm_mxfp4_e5m2_tile_kernel(
    TileProduct g, int tiles) {
    run_tiles<S, OutT, ROT>(g, tiles);
}

// Both gradient products of the error-only scheme in one grid, on tiles of one shape, with the rotation: a workgroup begins a tile of the
// second while others still hold one of the first, where two launches wait for the last of them.
template <class S>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu((S::OCC * S::kWaves + 3) / 4))) void gemm_mxfp4_e5m2_pair_kernel(
    TileProduct a, TileProduct b, int tiles_a, int tiles_b) {
    extern __shared__ uint32_t smem[];
    const uint32_t smem_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)smem;
    const int first_b = (tiles_a + 7) & ~7, t = (int)blockIdx.x;
    if (t >= tiles_a && (t < first_b || t - first_b >= tiles_b)) return;
    const bool second = t >= first_b;
    TileProduct g = a;   // uniform
    g.a_codes = second ? b.a_codes : a.a_codes;
    g.a_scales = second ? b.a_scales : a.a_scales;
    g.b_codes = second ? b.b_codes : a.b_codes;
    g.b_scales = second ? b.b_scales : a.b_scales;
    g.c = second ? b.c : a.c;
    g.mask = second ? b.mask : a.mask;
    g.M = second ? b.M : a.M;
    g.K = second ? b.K : a.K;
    g.rot_c = second ? b.rot_c : a.rot_c;
    g.out_f32 = second ? b.out_f32 : a.out_f32;
    g.b_wide = second ? b.b_wide : a.b_wide;
    tile_run<S, uint16_t, true>(g, second ? t - first_b : t, smem, smem_base);
}
template <class S, typename OutT, bool ROT = false>
hipError_t launch_tiles(const TileProduct& g, hipStream_t stream) {
    const auto kern = [] {
        if constexpr (S::kWideB) return gemm_mxfp4_e5m2_tile_kernel<S, OutT, ROT>;
        else return gemm_mxfp4_tn_tile_kernel<S, OutT, ROT>;
    }();
    static std::atomic<bool> lds_allowed[kMaxDevices];
    hipError_t e = allow_dynamic_lds(kern, S::kSmemBytes, lds_allowed);
    if (e != hipSuccess) return e;
    const int tiles = ((g.M + S::BM - 1) / S::BM) * ((g.N + S::BN - 1) / S::BN) * g.splits;
    // a grid that is a multiple of 8 so that tile t and t + grid land on the same XCD
    int grid = tiles < S::OCC * device_cus() ? tiles : S::OCC * device_cus();
    if (grid > 8 && grid < tiles) grid -= grid % 8;
    kern<<<dim3((unsigned)grid), dim3(S::kThreads), S::kSmemBytes, stream>>>(g, tiles);
    return hipGetLastError();
}

// Both gradient products of a layer in one grid, A's tiles first (the longer contraction's: they are on their way while B's pass
// through the chip).  Launched one after the other, each product ends in tiles that leave most of the chip idle, and a weight gradient
// of few tiles and many tokens is cut into K ranges whose partial sums travel through memory; here its whole tiles run beside the
// input gradient's.  us of a layer's backward pass on the GPU, two launches against one: 512 x 640 x 1920 25 -> 21, 2048^3 44 -> 37, 1824 x
// 2048 x 1408 39 -> 34, 16480 x 1728 x 640 (64 x 64 tiles of the weight gradient) 93 -> 87, 16384 x 1536 x 1536 124 -> 106, 13312 x 8704 x 640
// 220 -> 195.  What bounds it: as each product by itself, and for the last tiles of a long contraction its serial chain (0.25 us a step).
// Workgroups are dealt out by the hardware as CUs become free, which evens the two out.  B's tiles begin at a multiple of eight, so that both keep their runs of tiles to an XCD (xcd_run).
template <class SA, bool ROT_A, class SB, bool ROT_B>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SA::OCC < SB::OCC ? SA::OCC : SB::OCC))) void gemm_mxfp4_tn_pair_kernel(
    TileProduct a, TileProduct b, int tiles_a, int tiles_b) {
    static_assert(SA::kThreads == 256 && SB::kThreads == 256, "one size of workgroup");
    extern __shared__ uint32_t smem[];
    const uint32_t smem_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)smem;
    const int t = (int)blockIdx.x, first_b = (tiles_a + 7) & ~7;
    if (t < tiles_a) tile_run<SA, uint16_t, ROT_A>(a, t, smem, smem_base);
    else if (t >= first_b && t - first_b < tiles_b) tile_run<SB, uint16_t, ROT_B>(b, t - first_b, smem, smem_base);
}
template <class SA, bool ROT_A, class SB, bool ROT_B>
hipError_t launch_pair(const TileProduct& a, const TileProduct& b, hipStream_t stream) {
    const auto kern = gemm_mxfp4_tn_pair_kernel<SA, ROT_A, SB, ROT_B>;
    constexpr int kLds = SA::kSmemBytes > SB::kSmemBytes ? SA::kSmemBytes : SB::kSmemBytes;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    const hipError_t e = allow_dynamic_lds(kern, kLds, lds_allowed);
    if (e != hipSuccess) return e;
    const auto tiles = [](const TileProduct& g, int bm, int bn) { return ((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn); };
    const int ta = tiles(a, SA::BM, SA::BN), tb = tiles(b, SB::BM, SB::BN);
    kern<<<dim3((unsigned)(((ta + 7) & ~7) + tb)), dim3(256), kLds, stream>>>(a, b, ta, tb);
    return hipGetLastError();
}

// a plain product with one of those ends
template <class S, int AFTER>
__global__ __launch_bounds__(S::kThreads) __attribute__((amdgpu_waves_per_eu((S::OCC * S::kWaves + 3) / 4))) void gemm_mxfp4_tn_after_kernel(
    TileProduct g, TileAfter after, int tiles) {
    extern __shared__ uint32_t smem[];
    const uint32_t smem_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)smem;
    for (int t = (int)blockIdx.x; t < tiles; t += (int)gridDim.x) tile_run<S, uint16_t, false, AFTER>(g, t, smem, smem_base, after);
}
template <class S, int AFTER>
hipError_t launch_after(TileProduct g, const TileAfter& after, hipStream_t stream) {
    const auto kern = gemm_mxfp4_tn_after_kernel<S, AFTER>;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    const hipError_t e = allow_dynamic_lds(kern, S::kSmemBytes, lds_allowed);
    if (e != hipSuccess) return e;
    g.splits = 1;
    const int cols = AFTER == END_SWIGLU ? (int)padded_cols(g.N / 2) * 2 : g.N;
    const int tiles = ((g.M + S::BM - 1) / S::BM) * ((cols + S::BN - 1) / S::BN);
    int grid = tiles < S::OCC * device_cus() ? tiles : S::OCC * device_cus();
    if (grid > 8 && grid < tiles) grid -= grid % 8;
    kern<<<dim3((unsigned)grid), dim3(S::kThreads), S::kSmemBytes, stream>>>(g, after, tiles);
    return hipGetLastError();
}

using Tile256x128 = TileShape<256, 128, 128, 64, 3, 2>;
using Tile128x128 = TileShape<128, 128, 64, 64, 3, 3>;
// One more stage where no CU has a second workgroup, which would cover a request's latency.  Plain results, us with three stages and with four: 1024 x 4096^2
// 13.7 and 12.9, 768 x 4096 x 11008 36.0 and 32.3, 2048 x 1536 x 4096 12.3 and 11.3, 512 x 8192 x 1536 7.9 and 7.5, 1024 x 3072 x 8192 23.9 and 18.8, 1024 x 3456 x
// 640 5.6 either way.  Up to two workgroups to a CU neither gains (1280 x 4096 x 11008 46.0 and 46.4, 640 x 8192 x 1536 10.3 and 10.0, 1792 x 4096 x 11008 47.9 and
// 49.9).  Eight waves of 64 x 32 instead of four 13.8 -> 14.5 at 1024 x 4096^2, six stages 13.7: the next block's scales, asked for three steps ahead, hold a ring at
// four.
using Deep128x128 = TileShape<128, 128, 64, 64, 4, 2>;
using Tile128x64 = TileShape<128, 64, 64, 32, 4, 3>;
using Tile64x64 = TileShape<64, 64, 32, 32, 4, 4>;
using Tile64x32 = TileShape<64, 32, 32, 32, 6, 4>;
// with an eight-bit B.  4096^3 alone in us, scales step by step: 256x256 in 8 waves of 128 x 64, 3 stages 60; in 4 waves of 128 x 128 66; 256x128 73 to 84;
// 128x128 with 2 stages three times per CU 74, with 3 stages twice 81
using Wide256x256 = TileShape<256, 256, 128, 64, 3, 1, true>;
using Wide128x128 = TileShape<128, 128, 64, 64, 2, 3, true>;
using Wide128x64 = TileShape<128, 64, 64, 32, 3, 3, true>;
using Wide64x64 = TileShape<64, 64, 32, 32, 4, 3, true>;

}  // namespace

bool gemm_tile_serves(int64_t M, int64_t N, int64_t K, int a_tiled, int b_tiled, const void* c) {
    const bool k_ok = K % kBK == 0 || (K % kBK == 64 && K >= 192 && !a_tiled && !b_tiled);
    return M > 0 && N >= 8 && N % 8 == 0 && K > 0 && k_ok && M < (1 << 30) && N < (1 << 30) && K < (1 << 23) &&
           (reinterpret_cast<uintptr_t>(c) & 15) == 0;
}

// of the same N, alpha, Hadamard block and signs, on 256 x 256 tiles with formats chosen per block
bool gemm_wide_pair_serves(const TileProduct& a, const TileProduct& b) {
    const auto serves = [](const TileProduct& g) {
        return g.b_e5m2 && g.b_wide && g.mask && gemm_tile_serves(g.M, g.N, g.K, g.a_tiled, g.b_tiled, g.c) && g.K / kBK >= 4;
    };
    for (int w = 0; w < 4; ++w)
        if (a.signs.w[w] != b.signs.w[w]) return false;
    return serves(a) && serves(b) && a.N == b.N && a.alpha == b.alpha && a.hd == b.hd;
}
hipError_t gemm_wide_pair(TileProduct a, bool a_f32, TileProduct b, bool b_f32, hipStream_t stream) {
    using S = Wide256x256::Mixed;
    if (!gemm_wide_pair_serves(a, b)) return hipErrorInvalidValue;
    a.splits = b.splits = 1;
    a.out_f32 = a_f32;
    b.out_f32 = b_f32;
    const auto kern = gemm_mxfp4_e5m2_pair_kernel<S>;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    const hipError_t e = allow_dynamic_lds(kern, S::kSmemBytes, lds_allowed);
    if (e != hipSuccess) return e;
    const auto tiles = [](const TileProduct& g) { return ((g.M + S::BM - 1) / S::BM) * ((g.N + S::BN - 1) / S::BN); };
    const int ta = tiles(a), tb = tiles(b);
    kern<<<dim3((unsigned)(((ta + 7) & ~7) + tb)), dim3(S::kThreads), S::kSmemBytes, stream>>>(a, b, ta, tb);
    return hipGetLastError();
}

// a: the longer contraction; tiles of 128 x 128 or 64 x 64 either; scales in blocks (see gemm_tile), at least one of them rotated
bool gemm_tile_pair_serves(const TileProduct& a, int shape_a, const TileProduct& b, int shape_b) {
    const auto serves = [](const TileProduct& g, int shape) {
        return (shape == TILE_128x128 || shape == TILE_64x64) && !g.b_e5m2 && gemm_tile_serves(g.M, g.N, g.K, g.a_tiled, g.b_tiled, g.c) && g.K % kBK == 0 &&
               g.K / kBK >= 4 && ((reinterpret_cast<uintptr_t>(g.a_scales) | reinterpret_cast<uintptr_t>(g.b_scales)) & 3) == 0 &&
               (!g.mask || (g.hd <= (shape == TILE_64x64 ? 64 : 128) && g.N % g.hd == 0));
    };
    return (a.mask || b.mask) && serves(a, shape_a) && serves(b, shape_b);
}
hipError_t gemm_tile_pair(TileProduct a, int shape_a, bool a_f32, TileProduct b, int shape_b, bool b_f32, hipStream_t stream) {
    if (!gemm_tile_pair_serves(a, shape_a, b, shape_b)) return hipErrorInvalidValue;
    a.splits = b.splits = 1;
    a.out_f32 = a_f32;
    b.out_f32 = b_f32;
    const auto rotations = [&](auto sa, auto sb) {
        using SA = decltype(sa);
        using SB = decltype(sb);
        if (!a.mask) return launch_pair<SA, false, SB, true>(a, b, stream);
        return b.mask ? launch_pair<SA, true, SB, true>(a, b, stream) : launch_pair<SA, true, SB, false>(a, b, stream);
    };
    if (shape_a == TILE_64x64) return shape_b == TILE_64x64 ? rotations(Tile64x64{}, Tile64x64{}) : rotations(Tile64x64{}, Tile128x128{});
    return shape_b == TILE_64x64 ? rotations(Tile128x128{}, Tile64x64{}) : rotations(Tile128x128{}, Tile128x128{});
}

// tiled operands of either end: whole K steps, dwords of scales, offsets into all of B in 32 bits
bool gemm_tile_after_serves(const TileProduct& g) {
    return g.a_tiled && g.b_tiled && !g.b_e5m2 && !g.mask && gemm_tile_serves(g.M, g.N, g.K, 1, 1, g.c) && g.K % kBK == 0 && (int64_t)g.N * (g.K / 2) < (1ll << 31) &&
           ((reinterpret_cast<uintptr_t>(g.a_scales) | reinterpret_cast<uintptr_t>(g.b_scales)) & 3) == 0;
}
hipError_t gemm_tile_swiglu(const TileProduct& g, const TileAfter& after, hipStream_t stream) {
    if (!gemm_tile_after_serves(g) || g.N % 64) return hipErrorInvalidValue;
    return g.K / kBK >= 4 ? launch_after<Tile128x128, END_SWIGLU>(g, after, stream) : launch_after<Tile128x128::Narrow, END_SWIGLU>(g, after, stream);
}
hipError_t gemm_tile_rope(const TileProduct& g, const TileAfter& after, hipStream_t stream) {
    if (!gemm_tile_after_serves(g) || g.N != 3 * after.width || after.width % after.head_dim || after.head_dim % 8) return hipErrorInvalidValue;
    return g.K / kBK >= 4 ? launch_after<Tile128x128, END_ROPE>(g, after, stream) : launch_after<Tile128x128::Narrow, END_ROPE>(g, after, stream);
}

namespace {
// blocks of scales: every K range has at least four steps, all whole, and scale rows start at multiples of four bytes
bool scales_in_blocks(const TileProduct& g) {
    return g.K % kBK == 0 && g.K / kBK / g.splits >= 4 && ((reinterpret_cast<uintptr_t>(g.a_scales) | reinterpret_cast<uintptr_t>(g.b_scales)) & 3) == 0;
}
}  // namespace
bool gemm_tile_deep(const TileProduct& g) {
    return !g.b_e5m2 && !g.mask && scales_in_blocks(g) && (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128) * g.splits <= device_cus();
}

hipError_t gemm_tile(int shape, const TileProduct& g, int c_dtype, hipStream_t stream) {
    const bool blocks = scales_in_blocks(g);
    const auto run_plain = [&](auto s) {
        using S = decltype(s);
        return c_dtype == BF16 ? launch_tiles<S, uint16_t>(g, stream) : launch_tiles<S, float>(g, stream);
    };
    const auto run = [&](auto s) {
        using S = decltype(s);
        return c_dtype == BF16 && g.mask ? launch_tiles<S, uint16_t, true>(g, stream) : run_plain(s);
    };
    // 256 x 128 over fewer than eight steps: its two blocks of 384 rows are more in front of the first step than they save behind it
    // (4096 x 3456 x 640 in an evaluated model 14 us, 16 with blocks)
    const auto go = [&](auto s) {
        using S = decltype(s);
        const bool few = !S::kWideB && S::BM == 256 && g.K / kBK / g.splits < kShortTallSteps;
        if constexpr (S::kWideB)
            if (g.b_wide) return run(typename S::Mixed{});
        return blocks && !few ? run(s) : run(typename S::Narrow{});
    };
    if (g.b_e5m2) {
        switch (shape) {
            case WIDE_256x256: return go(Wide256x256{});
            case TILE_128x128: return go(Wide128x128{});
            case TILE_128x64: return go(Wide128x64{});
            default: return go(Wide64x64{});
        }
    }
    switch (shape) {
        case TILE_256x128: return go(Tile256x128{});
        case TILE_128x128: return gemm_tile_deep(g) ? run_plain(Deep128x128{}) : go(Tile128x128{});
        case TILE_128x64: return go(Tile128x64{});
        case TILE_64x64: return go(Tile64x64{});
        default: return go(Tile64x32{});
    }
}

}  // namespace qm
