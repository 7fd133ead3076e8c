// MXFP4 x MXFP4 "TN" GEMM on gfx950's block-scaled FP4 MFMA.
//
//   C[m, n] = alpha * sum_k A[m, k] * B[n, k]
//
// A: packed E2M1 codes [M, K/2] (element 2i in the low nibble of byte i) + E8M0 scales [M, K/32];
// B likewise with N rows.  Replaces the bf16 cuBLAS GEMMs the reference runs on de-quantized
// operands (src/models/quantization/backward.py:62,71-75,79-83) and the role of
// matmul_mxf4_bf16_tn in notebooks/benchmark_mxfp4.ipynb (CudaGemm).
//
// Instruction: v_mfma_scale_f32_32x32x64_f8f6f4 with both operands FP4.  Lane l of a wave feeds
// row (l % 32) of its operand with the 32 consecutive K values of one MX group (16 bytes) plus
// that group's E8M0 byte, so one MX group maps 1:1 onto one lane's share of the instruction.
// Within a K step of 128 (four MX groups per row) lane half h = l / 32 takes groups 2h and 2h+1
// in the two successive MFMAs; both operands use the same assignment, which is all the
// instruction needs.
//
// Kernels, picked by choose_product() at the end of the file:
//   gemm_mxfp4_tn_big4_kernel  any M >= 256, N a multiple of 64 and >= 256, K a multiple of 128 but not 640, whose last block of four
//                              K steps repeats (muted) up to three steps.
//                              Persistent, 256x256 macro tile, 4 waves x 128x128, operands global -> LDS directly into a
//                              4-stage ring, scales in blocks of four K steps, row-major or tiled code bytes, optional split-K.
//   gemm_tile.hip              tiles from 256x128 down to 64x32 for everything too small or too short for that one.
//   gemm_two.hip               256x192 tiles, two workgroups to a CU: plain bf16 results whose tiles fill the last round better so.
//   gemm_mxfp4_tn_kernel       any M, N and K % 32 == 0: 128x128 macro tile, 4 waves x 64x64, operands staged
//                              global -> registers -> LDS (rows padded from 64 to 80 bytes so the 16-byte fragment
//                              reads of 16 consecutive rows hit 64 distinct banks), double buffered.
// All keep fp32 accumulators in registers, use one barrier per K step and apply alpha in the epilogue.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gemm_common.h"
#include "shape_table.h"

namespace qm {

namespace {

constexpr int kPitchDw = 20;         // 80-byte LDS row pitch, in dwords

template <int BM, int BN>
struct GemmSmem {
    static constexpr int kStageDw = (BM + BN) * kPitchDw + BM + BN;  // codes + one scale dword per row
    static constexpr int kBytes = 2 * kStageDw * 4;
};

__device__ __forceinline__ uint32_t load_scale_dword(const uint8_t* __restrict__ scales, int64_t row_pitch,
                                                     int64_t row, int64_t rows, int64_t g0, int64_t groups,
                                                     bool aligned) {
    if (row >= rows) return 0u;
    const uint8_t* p = scales + row * row_pitch + g0;
    if (aligned && g0 + 4 <= groups) return *reinterpret_cast<const uint32_t*>(p);
    uint32_t s = 0u;
#pragma unroll
    for (int b = 0; b < 4; ++b)
        if (g0 + b < groups) s |= (uint32_t)p[b] << (8 * b);
    return s;
}

template <int BM, int BN, int WM, int WN, typename OutT>
__global__ __launch_bounds__(256) void gemm_mxfp4_tn_kernel(const uint8_t* __restrict__ a_codes,
                                                            const uint8_t* __restrict__ a_scales,
                                                            const uint8_t* __restrict__ b_codes,
                                                            const uint8_t* __restrict__ b_scales, int64_t M,
                                                            int64_t N, int64_t K, float alpha,
                                                            OutT* __restrict__ c) {
    static_assert((BM / WM) * (BN / WN) == 4, "four waves per workgroup");
    constexpr int TM = WM / 32, TN = WN / 32;
    constexpr int kAVec = BM * 4 / 256, kBVec = BN * 4 / 256;  // 16-byte loads per thread per step
    extern __shared__ uint32_t smem[];
    using S = GemmSmem<BM, BN>;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave / (BN / WN), wn = wave % (BN / WN);
    const int lrow = lane & 31, half = lane >> 5;

    const int64_t m0 = (int64_t)blockIdx.y * BM, n0 = (int64_t)blockIdx.x * BN;
    const int64_t code_pitch = K / 2, groups = K / 32;
    const bool scales_aligned = (groups % 4) == 0;
    const int nk = (int)((K + kBK - 1) / kBK);

    uint4 ra[kAVec], rb[kBVec];
    uint32_t rs = 0u;

    auto load_global = [&](int ks) {
        const int64_t kbyte0 = (int64_t)ks * kRowBytes;
#pragma unroll
        for (int i = 0; i < kAVec; ++i) {
            const int idx = tid + i * 256, row = idx >> 2, cv = idx & 3;
            ra[i] = make_uint4(0, 0, 0, 0);
            if (m0 + row < M && kbyte0 + cv * 16 < code_pitch)
                ra[i] = *reinterpret_cast<const uint4*>(a_codes + (m0 + row) * code_pitch + kbyte0 + cv * 16);
        }
#pragma unroll
        for (int i = 0; i < kBVec; ++i) {
            const int idx = tid + i * 256, row = idx >> 2, cv = idx & 3;
            rb[i] = make_uint4(0, 0, 0, 0);
            if (n0 + row < N && kbyte0 + cv * 16 < code_pitch)
                rb[i] = *reinterpret_cast<const uint4*>(b_codes + (n0 + row) * code_pitch + kbyte0 + cv * 16);
        }
        // threads [0, BM) fetch A's scale dwords, threads [BM, BM+BN) fetch B's (BM + BN <= 512 -> two rounds)
        rs = 0u;
        if (tid < BM) rs = load_scale_dword(a_scales, groups, m0 + tid, M, (int64_t)ks * 4, groups, scales_aligned);
        else if (tid - BM < BN) rs = load_scale_dword(b_scales, groups, n0 + (tid - BM), N, (int64_t)ks * 4, groups, scales_aligned);
    };
    uint32_t rs2 = 0u;  // second round of scale rows when BM + BN > 256
    auto load_global_scales2 = [&](int ks) {
        if constexpr (BM + BN > 256) {
            const int t2 = tid + 256;
            rs2 = 0u;
            if (t2 < BM) rs2 = load_scale_dword(a_scales, groups, m0 + t2, M, (int64_t)ks * 4, groups, scales_aligned);
            else if (t2 - BM < BN) rs2 = load_scale_dword(b_scales, groups, n0 + (t2 - BM), N, (int64_t)ks * 4, groups, scales_aligned);
        }
    };
    auto store_lds = [&](int buf) {
        uint32_t* sa = smem + buf * S::kStageDw;
        uint32_t* sb = sa + BM * kPitchDw;
        uint32_t* ss = sb + BN * kPitchDw;  // [BM] A scales then [BN] B scales
#pragma unroll
        for (int i = 0; i < kAVec; ++i) {
            const int idx = tid + i * 256, row = idx >> 2, cv = idx & 3;
            *reinterpret_cast<uint4*>(sa + row * kPitchDw + cv * 4) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < kBVec; ++i) {
            const int idx = tid + i * 256, row = idx >> 2, cv = idx & 3;
            *reinterpret_cast<uint4*>(sb + row * kPitchDw + cv * 4) = rb[i];
        }
        if (tid < BM + BN) ss[tid] = rs;
        if constexpr (BM + BN > 256) {
            if (tid + 256 < BM + BN) ss[tid + 256] = rs2;
        }
    };

    v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    load_global(0);
    load_global_scales2(0);
    store_lds(0);
    __syncthreads();

    for (int ks = 0; ks < nk; ++ks) {
        const int buf = ks & 1;
        if (ks + 1 < nk) {
            load_global(ks + 1);
            load_global_scales2(ks + 1);
        }
        const uint32_t* sa = smem + buf * S::kStageDw;
        const uint32_t* sb = sa + BM * kPitchDw;
        const uint32_t* ss = sb + BN * kPitchDw;
        uint32_t sca[TM], scb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) sca[i] = ss[wm * WM + i * 32 + lrow] >> (16 * half);
#pragma unroll
        for (int j = 0; j < TN; ++j) scb[j] = ss[BM + wn * WN + j * 32 + lrow] >> (16 * half);
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            v8i af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                uint4 q = *reinterpret_cast<const uint4*>(sa + (wm * WM + i * 32 + lrow) * kPitchDw + (2 * half + sub) * 4);
                af[i] = v8i{(int)q.x, (int)q.y, (int)q.z, (int)q.w, 0, 0, 0, 0};
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                uint4 q = *reinterpret_cast<const uint4*>(sb + (wn * WN + j * 32 + lrow) * kPitchDw + (2 * half + sub) * 4);
                bf[j] = v8i{(int)q.x, (int)q.y, (int)q.z, (int)q.w, 0, 0, 0, 0};
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if (sub == 0)
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(af[i], bf[j], acc[i][j], 4, 4, 0,
                                                                                     (int)sca[i], 0, (int)scb[j]);
                    else
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(af[i], bf[j], acc[i][j], 4, 4, 1,
                                                                                     (int)sca[i], 1, (int)scb[j]);
                }
        }
        if (ks + 1 < nk) store_lds(buf ^ 1);
        __syncthreads();
    }

    // epilogue: acc element e of a 32x32 tile is row 8*(e/4) + 4*half + e%4, column lane%32
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int64_t col = n0 + wn * WN + j * 32 + lrow;
            if (col >= N) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t row = m0 + wm * WM + i * 32 + 8 * (e / 4) + 4 * half + (e & 3);
                if (row >= M) continue;
                const float v = acc[i][j][e] * alpha;
                if constexpr (sizeof(OutT) == 2) c[row * N + col] = f32_to_bf16(v);
                else c[row * N + col] = v;
            }
        }
}


// ---- large-tile kernel: 256 x 256 macro tile, one wave per SIMD owning 128 x 128 -----------------
// Requires M % 256 == 0, N % 256 == 0, K % 128 == 0.
//
// Per K step of 128 a wave issues 32 MFMAs (2 sub-steps x 4 x 4 tiles) against 16 fragment reads of
// 16 bytes.  Operands go global -> LDS directly (global_load_lds_dwordx4: each wave instruction drops
// 64 x 16 B contiguously into LDS, no staging registers, no ds_write), into a ring of four stages, so
// a tile is requested three K steps before it is consumed.  LDS rows are 64 bytes; the 16-byte column
// of (row, c) is stored at c ^ ((row >> 2) & 3), applied on the global-address side of the load and on
// the fragment read, which keeps the 16-byte fragment reads of 32 consecutive rows off each other's banks.
constexpr int kBigM = 256, kBigN = 256;
constexpr int kStages = 4;
constexpr int kBOff = kBigM * kRowBytes;

struct SubFrags {
    uint4 a[4], b[4];  // one K sub-step (64 values): four A tiles, four B tiles
};

// frag_off = byte offset of this lane's 16 bytes for the wanted sub-step within tile 0 of its operand
__device__ __forceinline__ void big_read_sub(const uint8_t* __restrict__ stage, int a_off, int b_off, SubFrags& f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f.a[i] = *reinterpret_cast<const uint4*>(stage + a_off + i * 32 * kRowBytes);
        f.b[i] = *reinterpret_cast<const uint4*>(stage + kBOff + b_off + i * 32 * kRowBytes);
    }
}

// SWAP = false: A rows become result rows.  SWAP = true: B's rows (n) are fed as the MFMA's first operand and
// A's rows (m) as its second, so a lane ends up with 4 consecutive n of one m (contiguous in row-major C),
// which the bf16 epilogue packs into 8-byte LDS writes.
template <int SUB, bool SWAP, bool ZERO = false>
__device__ __forceinline__ void big_mfma_sub(const SubFrags& f, const uint32_t (&sca)[4], const uint32_t (&scb)[4],
                                             v16f (&acc)[4][4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const v8i av = v8i{(int)f.a[i].x, (int)f.a[i].y, (int)f.a[i].z, (int)f.a[i].w, 0, 0, 0, 0};
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            // back and forth over B's blocks: one operand changes from product to product instead of both at every fourth, which the
            // power limit returns as clock (8192 x 4096 x 11008 step 716 -> 714 us, 16384 x 4096^2 forward 161.0 -> 160.4; bit-identical)
            const int j = i & 1 ? 3 - jj : jj;
            const v8i bv = v8i{(int)f.b[j].x, (int)f.b[j].y, (int)f.b[j].z, (int)f.b[j].w, 0, 0, 0, 0};
            // ZERO: the tile's first product starts the accumulator from the constant 0 instead of reading it
            v16f cin;
            if constexpr (ZERO) {
#pragma unroll
                for (int e = 0; e < 16; ++e) cin[e] = 0.0f;
            } else {
                cin = acc[i][j];
            }
            if constexpr (SWAP)
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bv, av, cin, 4, 4, SUB, (int)scb[j], SUB, (int)sca[i]);
            else
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, cin, 4, 4, SUB, (int)sca[i], SUB, (int)scb[j]);
        }
    }
}

// ---- persistent variant: scales travel in blocks of four K steps ------------------------------------
// Fetching one scale dword per row per K step costs as many L2 requests as the codes themselves (each
// row's 4 bytes sit in a different cache line).  Here a wave-load brings 16 bytes per row = the scales of
// four K steps, into a small double-buffered LDS area behind the four code stages; a lane reads the
// scale vectors of its eight tile rows once per block and keeps them in registers.
constexpr int kCodeStageBytes = (kBigM + kBigN) * kRowBytes;            // 32 KiB
constexpr int kScaleAreaOff = kStages * kCodeStageBytes;                // 128 KiB
constexpr int kScaleBufBytes = (kBigM + kBigN) * 16;                    // 8 KiB per block of four K steps
constexpr int kEpiAreaOff = kScaleAreaOff + 2 * kScaleBufBytes;     // 144 KiB
constexpr int kEpiWaveBytes = 4096;                                  // 32 rows x 64 bf16 per wave
constexpr int kBig4SmemBytes = kEpiAreaOff + 4 * kEpiWaveBytes;      // 160 KiB

struct Big4Plan {
    const uint8_t* a;   // uniform: first code byte of this tile's A panel (row m0, K step 0)
    const uint8_t* b;
    const uint8_t* sa;  // uniform: first scale byte of this tile's A panel
    const uint8_t* sb;
    int kstep_a, kstep_b;   // bytes from one K step to the next: 64 row-major, 1024 tiled
    uint32_t voff_a[4];     // wave-load i of a K step, issued with instruction offset i * 1024, which moves its LDS destination
    uint32_t voff_b[4];     //   by as much (and the source back in place): row offset - i * 1024
    uint32_t lane_scales_a;   // this lane's byte offset inside a panel's scales: row wave*64 + lane
    uint32_t lane_scales_b;
    uint32_t lds_codes;     // wave-uniform LDS address of this wave's first A wave-load in stage 0
    uint32_t lds_scales;    // wave-uniform LDS address of this wave's A scale wave-load in buffer 0
};

__device__ __forceinline__ void big4_issue_codes(const Big4Plan& p, int stage, int ks) {
    const uint32_t base = p.lds_codes + stage * kCodeStageBytes;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        load_lds_b128_s(p.a + j * 1024 + ks * p.kstep_a, p.voff_a[j], base + j * 1024);
        load_lds_b128_s(p.b + j * 1024 + ks * p.kstep_b, p.voff_b[j], base + kBOff + j * 1024);
    }
}
// soff: byte offset, within a row's scales, of the 16 bytes (four K steps) to request
__device__ __forceinline__ void big4_issue_scales(const Big4Plan& p, int soff, int buf) {
    const uint32_t base = p.lds_scales + buf * kScaleBufBytes;
    load_lds_b128_s(p.sa + soff, p.lane_scales_a, base);
    load_lds_b128_s(p.sb + soff, p.lane_scales_b, base + kBigM * 16);
}

// The LDS destination of a global->LDS load is M0 + the instruction's offset + lane * 16, and the same offset is added
// to the source address: with the lane offsets of Big4Plan::voff_* one M0 value serves the four wave-loads of an
// operand, and the loads themselves are single instructions between the MFMAs (every instruction a wave issues costs
// it four to five cycles, and a K step has only 32 cycles per MFMA to hide them in).
__device__ __forceinline__ void set_lds_dma_base(uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" ::"s"(lds_base));
}
template <int I>
__device__ __forceinline__ void load_lds_b128_m0(const uint8_t* base, uint32_t lane_off) {
    asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" ::"v"(lane_off), "s"(base), "i"(I * 1024) : "memory");
}

struct ScaleRegs {
    uint4 a[4], b[4];  // per tile: the row's scale dwords of the block's four K steps
};
__device__ __forceinline__ void big4_read_scales(const uint8_t* __restrict__ sbuf, int a_off, int b_off, ScaleRegs& r) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r.a[i] = *reinterpret_cast<const uint4*>(sbuf + a_off + i * 32 * 16);
        r.b[i] = *reinterpret_cast<const uint4*>(sbuf + kBigM * 16 + b_off + i * 32 * 16);
    }
}
template <int Q>
__device__ __forceinline__ uint32_t pick(const uint4& v) {
    return Q == 0 ? v.x : (Q == 1 ? v.y : (Q == 2 ? v.z : v.w));
}


struct Big4State {
    SubFrags f0, f1;
    ScaleRegs sr;
};

// One K step of the flat (tile, K step) stream; the step's index in its tile is congruent to Q mod 4, so
// the ring stage it consumes is Q.  `lks` is the K step (of the tile `plan` points at) whose codes it
// requests into the stage it has just freed, `soff` (Q = 0 only) the byte offset of the scale block it requests;
// `sw` = 16, or 0 for a step whose scale bytes are to read as zero (2^-127: its products vanish); `par` selects the
// scale buffer the current block lives in.
template <int Q, bool SWAP, bool FIRST = false, int EXTRA = 0>
__device__ __forceinline__ void big4_step(const Big4Plan& plan, uint8_t* smem_bytes, int lks, int soff, int sw, int par, int a_off0,
                                          int a_off1, int b_off0, int b_off1, int a_sc_off, int b_sc_off, int sh,
                                          Big4State& st, v16f (&acc)[4][4]) {
    const uint8_t* cur = smem_bytes + Q * kCodeStageBytes;
    const uint8_t* nxt = smem_bytes + ((Q + 1) & 3) * kCodeStageBytes;
    // the lane half's two scale bytes of this step: bits [sh, sh + 16) of the row's dword; sw = 0 mutes the step
    const auto two = [&](const uint4& v) { return __builtin_amdgcn_ubfe(pick<Q>(v), (uint32_t)sh, (uint32_t)sw); };
    const uint32_t sca[4] = {two(st.sr.a[0]), two(st.sr.a[1]), two(st.sr.a[2]), two(st.sr.a[3])};
    const uint32_t scb[4] = {two(st.sr.b[0]), two(st.sr.b[1]), two(st.sr.b[2]), two(st.sr.b[3])};
    big_read_sub(cur, a_off1, b_off1, st.f1);
    big_mfma_sub<0, SWAP, FIRST>(st.f0, sca, scb, acc);
    QM_SCHED_PAIR(0x100, 8)
    __builtin_amdgcn_sched_barrier(0);
    // loads younger than the codes of the next step: the codes of the two steps after it (16) and, for Q = 1, 2,
    // the two scale loads issued since; for Q = 3 the scale block read below is older than those and must be in
    // EXTRA: requests of another kind issued since the awaited stage's (the fused epilogue's mask words, which a tile
    // requests at its first K step and which may stay pending through its first three)
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(((Q == 1 || Q == 2) ? 18 : 16) + EXTRA));
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (Q == 3) big4_read_scales(smem_bytes + kScaleAreaOff + (par ^ 1) * kScaleBufBytes, a_sc_off, b_sc_off, st.sr);
    // one quarter of the step's requests and fragment reads per four MFMAs (same issue order as the clumped form)
    {
        const uint32_t base = plan.lds_codes + Q * kCodeStageBytes;
        if constexpr (Q == 3) __builtin_amdgcn_sched_barrier(0);
        const uint8_t* src_a = plan.a + lks * plan.kstep_a;  // uniform: this wave's panel rows, K step lks
        const uint8_t* src_b = plan.b + lks * plan.kstep_b;
        set_lds_dma_base(base);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const v8i av = v8i{(int)st.f1.a[i].x, (int)st.f1.a[i].y, (int)st.f1.a[i].z, (int)st.f1.a[i].w, 0, 0, 0, 0};
            const auto products = [&](int j0, int j1) {
#pragma unroll
                for (int jj = j0; jj < j1; ++jj) {
                    const int j = i & 1 ? 3 - jj : jj;
                    const v8i bv = v8i{(int)st.f1.b[j].x, (int)st.f1.b[j].y, (int)st.f1.b[j].z, (int)st.f1.b[j].w, 0, 0, 0, 0};
                    if constexpr (SWAP)
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bv, av, acc[i][j], 4, 4, 1, (int)scb[j], 1, (int)sca[i]);
                    else
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, acc[i][j], 4, 4, 1, (int)sca[i], 1, (int)scb[j]);
                }
            };
            // per four MFMAs: two fragment reads of the next stage and two of the step's eight wave-loads (A's four,
            // then B's four behind a second M0 value)
            st.f0.a[i] = *reinterpret_cast<const uint4*>(nxt + a_off0 + i * 32 * kRowBytes);
            if (i == 0) load_lds_b128_m0<0>(src_a, plan.voff_a[0]);
            if (i == 1) load_lds_b128_m0<2>(src_a, plan.voff_a[2]);
            if (i == 2) { set_lds_dma_base(base + kBOff); load_lds_b128_m0<0>(src_b, plan.voff_b[0]); }
            if (i == 3) load_lds_b128_m0<2>(src_b, plan.voff_b[2]);
            st.f0.b[i] = *reinterpret_cast<const uint4*>(nxt + kBOff + b_off0 + i * 32 * kRowBytes);
            if (i == 0) load_lds_b128_m0<1>(src_a, plan.voff_a[1]);
            if (i == 1) load_lds_b128_m0<3>(src_a, plan.voff_a[3]);
            if (i == 2) load_lds_b128_m0<1>(src_b, plan.voff_b[1]);
            if (i == 3) load_lds_b128_m0<3>(src_b, plan.voff_b[3]);
            if constexpr (Q == 0) {
                if (i == 3) big4_issue_scales(plan, soff, par ^ 1);
            }
            products(0, 4);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// bf16 epilogue (operand roles swapped: a lane's accumulator quads run along n).  Eight passes of 32 rows x 64
// columns per wave through a private 4 KiB LDS stage outside the operand ring, so the next tile's operands
// keep streaming in underneath; 16-byte chunks are XOR-swizzled by row so that writes and reads spread over
// all banks.
// ROT (a Hadamard block, 32, 64 or 128; 0: none): the masked inverse Hadamard rotation of the layer's backward pass applied to the tile before it
// is stored: out[m][n'] = c * sum_n (bf16(alpha * acc[m][n]) * keep[m][n]) * S[n'][n] * sign[n], S the 32 x 32 Sylvester
// matrix.  With the operand roles swapped a lane holds 16 of a group's 32 n for one m, which is the layout the bf16
// matrix instruction reads its second operand in (k along the registers, column = lane % 32); its first operand is the
// +-1 matrix, rebuilt per tile from the sign word.  The sums are fp32 sums of bf16 values in the instruction's order
// (the stand-alone kernel adds them as a butterfly), the factor c and the final rounding are the same.
// Blocks of 64 and 128 are sums and differences of those of 32 in the lane's own registers: 32 or 128 vector additions a pass, which
// makes this kernel serve what 128 x 128 tiles with lane exchanges did.  us per training step, hd 128: 8192 x 4096^2 335 -> 306,
// 8192 x 1536 x 4608 with an fp32 weight 204 -> 192, 6912 x 7168 x 3968 477 -> 440; hd 64: 8192 x 4096^2 332 -> 302.
struct RotEpilogue {
    const uint8_t* mask;  // [M][N / 8] clip-mask bits, bit n % 8 of byte n / 8
    uint32_t signs;       // bit n: column n of every 32 of the Hadamard block negated
    float c;              // block^-1/2, rounded to the scale dtype
};
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// WIDE: the rotated, bf16-rounded result leaves widened to fp32 (the weight gradient of an fp32 weight), 32 columns at a time through
// the same 4 KiB, whole 128-byte lines out.
template <int ROT = 0, bool RAGGED = false, bool WIDE = false, bool UNIT = false>
__device__ __forceinline__ void big4_epilogue_bf16(v16f (&acc)[4][4], float alpha, void* __restrict__ c, int64_t m0,
                                                   int64_t n0, int64_t N, int wm, int wn, int wave, int lane_in,
                                                   uint8_t* smem_bytes, int rows_valid, int cols_valid,
                                                   [[maybe_unused]] const RotEpilogue& rot, [[maybe_unused]] const u32x4 (&keep)[4],
                                                   [[maybe_unused]] bool keep_shifted) {
    static_assert(ROT || !WIDE, "plain fp32 results have an epilogue of their own");
    constexpr int kOut = WIDE ? 4 : 2;   // bytes per result
    constexpr int kSide = ROT == 128 ? 4 : 2;   // blocks of 32 columns per pass
    // The opaque copy keeps the address arithmetic below inside the (rarely executed) epilogue instead of being
    // hoisted out of the K loop, where it would hold dozens of registers across the MFMA schedule.
    // the lane index straight from the hardware, so that no copy of it has to stay alive through the K loop
    (void)lane_in;
    int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));
    const int lrow = lane & 31, half = lane >> 5;
    uint8_t* region = smem_bytes + kEpiAreaOff + wave * kEpiWaveBytes;
    const int chunk = lane & 7, rsub = lane >> 3;
    uint8_t* wr = region + lrow * 128 + half * 8;
    const int wsw = (lrow & 7) * 16;
    const uint8_t* rd = region + rsub * 128 + ((chunk ^ rsub) * 16);  // rows rsub + 8k share rsub's swizzle
    const int64_t pitch8 = N * 8 * kOut;                             // eight rows
    uint8_t* out = static_cast<uint8_t*>(c) + ((m0 + wm * 128 + rsub) * N + n0 + wn * 128) * kOut + chunk * 16;
    // rows [32 i, 32 i + 32) of the wave's tile, the 128 bytes of each that the stage holds, from byte `col` of its columns on
    const auto put_rows = [&](int i, int col) {
#pragma unroll
        for (int r8 = 0; r8 < 4; ++r8)
            if (!RAGGED || i * 32 + r8 * 8 + rsub < rows_valid) {
                const uint4 v = *reinterpret_cast<const uint4*>(rd + r8 * 1024);
                // streaming store: the tile is not read again by this kernel, and keeping it out of the L2 leaves the
                // operand panels there (measured: -1.3 % on the product alone, -3 % on the whole layer step)
                typedef uint32_t u4v __attribute__((ext_vector_type(4)));
                __builtin_nontemporal_store(u4v{v.x, v.y, v.z, v.w}, reinterpret_cast<u4v*>(out + r8 * pitch8 + col));
            }
    };
    // ROT: `keep[i]` holds the four mask words of the lane's row in block row i (one per 32 x 32 block: its group of 32 n),
    // requested at the tile's first K step.  The +-1 matrix: lane (n' = lane % 32, half h) holds, for instruction q,
    // S[n'][n] sign[n] at n = 8 (2 q + rho) + 4 h + e
    [[maybe_unused]] v8bf hmat[2];
    // a factor c that bf16 holds exactly (the bf16 scale dtype) rides in the matrix entries: the products stay exact in fp32
    // and the multiplication after the sums falls away
    [[maybe_unused]] const bool c_in_matrix = ROT && (f2u(rot.c) & 0xffffu) == 0u;
    if constexpr (ROT) {
        const uint32_t one = c_in_matrix ? f2u(rot.c) >> 16 : 0x3f80u;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            uint32_t w[4];
#pragma unroll
            for (int pr = 0; pr < 4; ++pr) {   // pair pr: rho = pr / 2, e = 2 (pr % 2), +1
                uint32_t bits = 0u;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int n = 8 * (2 * q + pr / 2) + 4 * half + 2 * (pr & 1) + k;
                    const uint32_t neg = ((uint32_t)__builtin_popcount((uint32_t)(lrow & n)) ^ (rot.signs >> n)) & 1u;
                    bits |= (one | (neg << 15)) << (16 * k);
                }
                w[pr] = bits;
            }
            hmat[q] = __builtin_bit_cast(v8bf, u32x4{w[0], w[1], w[2], w[3]});
        }
    }
    acc_settle();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int jp = 0; jp < 4 / kSide; ++jp) {
            if (i * 32 >= rows_valid || jp * kSide * 32 >= cols_valid) continue;  // uniform: this pass lies outside the matrix
            if constexpr (!ROT) {
#pragma unroll
                for (int jj = 0; jj < 2; ++jj) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const v16f& t = acc[i][2 * jp + jj];
                        const float t0 = acc_read(t[4 * b]), t1 = acc_read(t[4 * b + 1]), t2 = acc_read(t[4 * b + 2]), t3 = acc_read(t[4 * b + 3]);
                        const v2bf p0 = __builtin_convertvector(UNIT ? v2f{t0, t1} : v2f{t0 * alpha, t1 * alpha}, v2bf);
                        const v2bf p1 = __builtin_convertvector(UNIT ? v2f{t2, t3} : v2f{t2 * alpha, t3 * alpha}, v2bf);
                        *reinterpret_cast<uint2*>(wr + (((jj * 4 + b) * 16) ^ wsw)) =
                            make_uint2(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1));
                    }
                }
                put_rows(i, jp * 128);
            } else {
                // Both blocks of the pass go through the matrix pipe before either result is read: the second block's
                // conversion and masking run while the first block's instructions are in flight (the opaque copies below
                // keep the read-out of the results behind both blocks' matrix instructions).  Per tile 15.9 k -> 14.7 k cycles.
                v16f r[kSide];
#pragma unroll
                for (int jj = 0; jj < kSide; ++jj) {
                    const v16f& t = acc[i][kSide * jp + jj];
                    // the block rounded to bf16 and masked: register pair 2 b + k holds n = 8 b + 4 half + 2 k, + 1
                    // the block's mask word: word j of the row's four, or word j + 2 where the wave requested the row's last
                    // 16 bytes (its columns hang over the edge of N; blocks 2 and 3 are then outside and skipped)
                    const uint32_t kword = keep_shifted ? keep[i][(kSide * jp + jj + 2) & 3] : keep[i][kSide * jp + jj];
                    const uint32_t kw = kword >> (4 * half);
                    uint32_t pk[8];
#pragma unroll
                    for (int b = 0; b < 4; ++b)
#pragma unroll
                        for (int k = 0; k < 2; ++k) {
                            const float t0 = acc_read(t[4 * b + 2 * k]), t1 = acc_read(t[4 * b + 2 * k + 1]);
                            const uint32_t p = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{t0 * alpha, t1 * alpha}, v2bf));
                            const uint32_t lo = (uint32_t)__builtin_amdgcn_sbfe((int)kw, 8 * b + 2 * k, 1);       // 0 or ~0
                            const uint32_t hi = (uint32_t)__builtin_amdgcn_sbfe((int)kw, 8 * b + 2 * k + 1, 1);
                            pk[2 * b + k] = p & ((lo & 0xffffu) | (hi & 0xffff0000u));
                        }
                    v16f z;
#pragma unroll
                    for (int e = 0; e < 16; ++e) z[e] = 0.0f;
                    z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hmat[0], __builtin_bit_cast(v8bf, u32x4{pk[0], pk[1], pk[2], pk[3]}), z, 0, 0, 0);
                    r[jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hmat[1], __builtin_bit_cast(v8bf, u32x4{pk[4], pk[5], pk[6], pk[7]}), z, 0, 0, 0);
                }
                if constexpr (ROT > 32) {
                    // the block of 64 or 128 is Sylvester's matrix of order 2 or 4 over these of order 32: sums and differences
#pragma unroll
                    for (int jj = 0; jj < kSide; ++jj) asm volatile("" : "+v"(r[jj]));
#pragma unroll
                    for (int st = 1; st < ROT / 32; st *= 2)
#pragma unroll
                        for (int jj = 0; jj < kSide; ++jj)
                            if (!(jj & st)) {
#pragma unroll
                                for (int e = 0; e < 16; ++e) {
                                    const float u = r[jj][e], v = r[jj + st][e];
                                    r[jj][e] = u + v;
                                    r[jj + st][e] = u - v;
                                }
                            }
                }
                const auto emit = [&](auto scaled) {
#pragma unroll
                    for (int jj = 0; jj < kSide; ++jj) {
                        if constexpr (ROT == 32) asm volatile("" : "+v"(r[jj]));
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            float q[4];
#pragma unroll
                            for (int e = 0; e < 4; ++e) q[e] = decltype(scaled)::value ? r[jj][4 * b + e] * rot.c : r[jj][4 * b + e];
                            const uint32_t p0 = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{q[0], q[1]}, v2bf));
                            const uint32_t p1 = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{q[2], q[3]}, v2bf));
                            if constexpr (WIDE)
                                *reinterpret_cast<uint4*>(region + lrow * 128 + (((2 * b + half) * 16) ^ wsw)) =
                                    make_uint4(p0 << 16, p0 & 0xffff0000u, p1 << 16, p1 & 0xffff0000u);
                            else
                                *reinterpret_cast<uint2*>(wr + ((((jj & 1) * 4 + b) * 16) ^ wsw)) = make_uint2(p0, p1);
                        }
                        // the region is private to the wave; LDS operations of one wave complete in order
                        if constexpr (WIDE) {   // N is a multiple of 64: both blocks of the pass are inside
                            __builtin_amdgcn_wave_barrier();
                            put_rows(i, (kSide * jp + jj) * 128);
                            __builtin_amdgcn_wave_barrier();
                        } else if (jj & 1) {
                            put_rows(i, (kSide * jp + jj) / 2 * 128);
                        }
                    }
                };
                if (c_in_matrix) emit(std::false_type{});
                else emit(std::true_type{});
            }
            // keeps the passes apart: a scheduler that reads many passes' accumulators into vector registers ahead of time
            // pushes the K loop's live values out to scratch memory, and their reloads wait for every operand load in flight
            __builtin_amdgcn_sched_barrier(0);
        }
        out += 4 * pitch8;
    }
}

// Measurement aid (the STAMP instantiation of the kernel below): the shader clock at a workgroup's entry, at the start of
// its tile loop, and after every tile's K loop and epilogue, kPhaseStamps values per workgroup at the kernel's `stamps`
// argument (which the production instantiation never reads).
constexpr int kPhaseStamps = 32;  // entry, loop start, then (K loop end, epilogue end) of up to 15 tiles
__device__ __forceinline__ unsigned long long shader_clock() {
    unsigned long long t;
    // the counter arrives like a scalar load: without the wait the registers it lands in may be reused before it does
    asm volatile("s_memtime %0\n\ts_waitcnt lgkmcnt(0)" : "=s"(t));
    return t;
}

// Two products in one grid: the gradients of a layer, gx = Q(e) Q(W^T)^T [T x I, over O] and gw = Q(e^T) Q(x^T)^T [O x I, over T].  They
// share nothing but N; the one with more K steps comes first and is "the long one".  Launched one after the other each ends in a
// round of tiles that fills part of the chip, or is cut into K ranges whose partial sums travel through memory; together the tiles
// of one fill the gaps of the other.  Every XCD has a contiguous run of either product's tiles, its W = grid / 8 workgroups take the
// long ones in turn, then `rounds` short ones each, and those that had one long tile fewer take the short ones that are left:
// the host picks `rounds` so that all end together.  What bounds it is what bounds the kernel with one product (the power limit: 3.4 to
// 4.1 PFLOP/s); figures at pair_margin().
struct Big4Other {   // the short product; the long one is the kernel's first arguments
    const uint8_t* a_codes;
    const uint8_t* a_scales;
    const uint8_t* b_codes;
    const uint8_t* b_scales;
    void* c;
    RotEpilogue rot;
    int M, K;
    int rounds;
    int kind, long_kind;   // Big4Result of the short and of the long product
};
struct Big4NoOther {};
enum Big4Result : int { BIG4_PLAIN = 1, BIG4_ROTATED = 2, BIG4_WIDE = 4 };   // bf16, with the rotation, with it and widened to fp32

// Persistent: the grid is one workgroup per CU (or fewer); each workgroup walks tiles bid, bid + grid, ... as one
// flat stream of K steps.  The loads that refill a freed ring stage simply continue into the next tile, so the
// pipeline never drains between tiles and the epilogue runs while the next tile's first four stages arrive.
// RAGGED: M is not a multiple of 64 (an instantiation of its own: the row tests cost the others 2 to 8 % in registers).
// UNIT: alpha is 1 (a layer's forward product, bf16 result): 256 multiplications less among the epilogue's ~770 vector instructions a
// tile, which nothing overlaps.  Whole inference calls: 16384 x 1536 x 8192 125.8 -> 123.0 us, 16384 x 1536 x 4608 80.6 -> 79.3, 8192 x 4096 x
// 11008 194.2 -> 192.8; 8192 x 4096 x 4096 the same.
// PAIR: two products (Big4Other), tiled operands; the sum of the kinds of result that they have.
template <typename OutT, bool STAMP = false, int ROT = 0, bool RAGGED = false, int PAIR = 0, bool UNIT = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_mxfp4_tn_big4_kernel(
    const uint8_t* __restrict__ a_codes, const uint8_t* __restrict__ a_scales, const uint8_t* __restrict__ b_codes,
    const uint8_t* __restrict__ b_scales, int M, int N, int K, float alpha, OutT* __restrict__ c, int a_tiled,
    int b_tiled, int splits, int late, [[maybe_unused]] unsigned long long* __restrict__ stamps,
    [[maybe_unused]] RotEpilogue rot = RotEpilogue{}, [[maybe_unused]] std::conditional_t<PAIR != 0, Big4Other, Big4NoOther> other = {}) {
    static_assert(!ROT || sizeof(OutT) == 2, "the fused inverse rotation is part of the bf16 epilogue");
    static_assert(!PAIR || (ROT && !STAMP && (PAIR & (BIG4_ROTATED | BIG4_WIDE))), "a pair without any rotation holds mask words that nothing reads");
    extern __shared__ uint32_t smem[];
    uint8_t* smem_bytes = reinterpret_cast<uint8_t*>(smem);
    const uint32_t smem_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t*)smem;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    [[maybe_unused]] int stamps_taken = 0;
    const auto stamp = [&]() {
        if constexpr (STAMP) {
            const unsigned long long now = shader_clock();
            if (tid == 0 && stamps_taken < kPhaseStamps) stamps[(size_t)blockIdx.x * kPhaseStamps + stamps_taken] = now;
            ++stamps_taken;
        }
    };
    stamp();
    // wave-uniform by construction; saying so keeps everything derived from it (tile corners, edge tests, the epilogue's
    // base addresses) in scalar registers
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int lrow = lane & 31, half = lane >> 5;
    const int tiles_m = (M + kBigM - 1) / kBigM, tiles_n = (N + kBigN - 1) / kBigN, total = tiles_m * tiles_n;
    const int code_pitch = K / 2, groups = K / 32;
    // Split K: a work item is (tile, K range); with splits > 1 (fp32 instantiation only) item (t, s) covers K steps
    // [s * nk, (s + 1) * nk) and stores its partial sums, unscaled, into slab s of c = [splits][M][N].
    // K steps per work item.  The pipeline walks blocks of four steps.  When K is not a multiple of 512 (one work item
    // then) the last block covers the row's final four steps, and those of them that the block before has already
    // added are muted: their scale bytes read as zero (2^-127 each), so every product is below the smallest fp32
    // denormal and adds an exact zero.  No request leaves the operand's rows.
    const int nk_real = K / kBK / splits;
    const int nk = (nk_real + 3) & ~3;
    const int muted = nk - nk_real;  // steps of the last block that repeat the block before (0: K steps in whole blocks)
    const int total_items = total * splits;
    const int stride = (int)gridDim.x;

    const int swz = (lrow >> 2) & 3;
    const int a_off0 = (wm * 128 + lrow) * kRowBytes + (((2 * half) ^ swz) * 16);
    const int a_off1 = (wm * 128 + lrow) * kRowBytes + (((2 * half + 1) ^ swz) * 16);
    const int b_off0 = (wn * 128 + lrow) * kRowBytes + (((2 * half) ^ swz) * 16);
    const int b_off1 = (wn * 128 + lrow) * kRowBytes + (((2 * half + 1) ^ swz) * 16);
    const int a_sc_off = (wm * 128 + lrow) * 16, b_sc_off = (wn * 128 + lrow) * 16;
    const int sh = 16 * half;

    Big4Plan plan;
    plan.lds_codes = (uint32_t)__builtin_amdgcn_readfirstlane((int)(smem_base + wave * 4096));
    plan.lds_scales = (uint32_t)__builtin_amdgcn_readfirstlane((int)(smem_base + kScaleAreaOff + wave * 1024));
    const uint32_t row16 = 16u * (uint32_t)code_pitch;   // 16 rows are 8 K bytes in either layout, 512 <= K < 2^26: 63 rows stay below 2^31
    // the offsets of clamped rows may fall below i * 1024: RAGGED takes them from a base that much further back
    constexpr uint32_t kLoadBias = RAGGED ? 3 * 1024 : 0;
    // source of this lane in wave-load i: row 16 i + lane / 4 of the wave's 64 (at most `last`), swizzled 16-byte column
    const auto lane_source = [&](int i, int last, int tiled, uint32_t rows16, int pitch) {
        const int prow = lane >> 2, pcv = (lane & 3) ^ ((prow >> 2) & 3);
        int r = 16 * i + prow;
        r = r < last ? r : last;
        const uint32_t off = tiled ? (uint32_t)(r >> 4) * rows16 + (uint32_t)(r & 15) * 64u : (uint32_t)r * (uint32_t)pitch;
        return off + pcv * 16 + kLoadBias - 1024u * i;
    };
    plan.kstep_a = a_tiled ? 1024 : kRowBytes;
    plan.kstep_b = b_tiled ? 1024 : kRowBytes;
    plan.lane_scales_a = plan.lane_scales_b = (uint32_t)(lane * groups);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        plan.voff_a[i] = lane_source(i, 63, a_tiled, row16, code_pitch);
        plan.voff_b[i] = lane_source(i, 63, b_tiled, row16, code_pitch);
    }
    const int wave_u = wave;
    int load_tm, load_tn, load_split;  // work item the load stream is in
    [[maybe_unused]] bool load_short = false;
    // the panels of the tile at (load_tm, load_tn) of a product
    const auto plan_panels = [&](const uint8_t* ac, const uint8_t* as, const uint8_t* bc, const uint8_t* bs, int rows, int pitch, int64_t k0) {
        // N, and but for RAGGED M, is a multiple of 64: a wave's 64-row share of a panel is inside the matrix or outside it as a
        // whole; an outside share reads the matrix's last 64 rows instead (its products are dropped by the epilogue).
        // RAGGED: A's rows past the end read the last row (of the last block of 16 in a tiled operand).
        const int g = pitch / 16;
        int64_t m0 = (int64_t)load_tm * kBigM + wave_u * 64, n0 = (int64_t)load_tn * kBigN + wave_u * 64;
        m0 = m0 < rows ? m0 : RAGGED ? (int64_t)((rows - 1) & ~63) : (int64_t)rows - 64;
        n0 = n0 < N ? n0 : (int64_t)N - 64;
        plan.a = ac + m0 * pitch + k0 * plan.kstep_a - kLoadBias;
        plan.b = bc + n0 * pitch + k0 * plan.kstep_b - kLoadBias;
        if constexpr (RAGGED || PAIR) {   // otherwise the lane offsets never change
            const int last = RAGGED ? rows - 1 - (int)m0 : 63, last_code = a_tiled ? last | 15 : last;
            const uint32_t rows16 = 16u * (uint32_t)pitch;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                plan.voff_a[i] = lane_source(i, last_code, a_tiled, rows16, pitch);
                if constexpr (PAIR) plan.voff_b[i] = lane_source(i, 63, b_tiled, rows16, pitch);
            }
            plan.lane_scales_a = (uint32_t)((lane < last ? lane : last) * g);
            if constexpr (PAIR) plan.lane_scales_b = (uint32_t)(lane * g);
        }
        plan.sa = as + m0 * g + k0 * 4;
        plan.sb = bs + n0 * g + k0 * 4;
    };
    // PAIR: the next of this workgroup's tiles, the `taken`-th; false behind the last one
    [[maybe_unused]] int taken = 0;
    const auto next_of_pair = [&]() -> bool {
        if constexpr (PAIR != 0) {
            const int W = (int)gridDim.x >> 3, j = (int)blockIdx.x >> 3, xcd = (int)blockIdx.x & 7, back = 7 - xcd;
            const int short_tiles = (other.M + kBigM - 1) / kBigM * tiles_n;
            const int longs = (total >> 3) + (xcd < (total & 7) ? 1 : 0), shorts = (short_tiles >> 3) + (back < (short_tiles & 7) ? 1 : 0);
            const int heavy = longs % W;   // workgroups with a long tile more than the others
            int at = j + W * taken;
            load_short = at >= longs;
            if (load_short) {
                const int r = taken - longs / W - (j < heavy ? 1 : 0);
                if (r >= other.rounds && heavy && j < heavy) return false;
                at = r < other.rounds || !heavy ? j + W * r : W * other.rounds + (j - heavy) + (W - heavy) * (r - other.rounds);
                if (at >= shorts) return false;
                // the short product's extra tiles go to the XCDs that have none of the long one's
                at += back * (short_tiles >> 3) + (back < (short_tiles & 7) ? back : short_tiles & 7);
                tile_of_run(at, (other.M + kBigM - 1) / kBigM, tiles_n, load_tm, load_tn);
            } else {
                at += xcd * (total >> 3) + (xcd < (total & 7) ? xcd : total & 7);
                tile_of_run(at, tiles_m, tiles_n, load_tm, load_tn);
            }
            ++taken;
            if (load_short) plan_panels(other.a_codes, other.a_scales, other.b_codes, other.b_scales, other.M, other.K / 2, 0);
            else plan_panels(a_codes, a_scales, b_codes, b_scales, M, code_pitch, 0);
        }
        return true;
    };
    auto plan_tile = [&](int item) {
        const int r = xcd_run(item, total_items);
        load_split = r / total;
        tile_of_run(r - load_split * total, tiles_m, tiles_n, load_tm, load_tn);
        plan_panels(a_codes, a_scales, b_codes, b_scales, M, code_pitch, (int64_t)load_split * nk_real);   // from the item's first K step
    };

    // Short contractions: every other group of eight workgroups (one per XCD) starts `late` x 1024 cycles late -- about the
    // length of an epilogue -- so that half of an XCD's CUs convert and store their tiles while the other half multiply.
    // Left alone the CUs can fall into step, and then every tile boundary is a burst of 33 MB of stores during which no CU
    // multiplies; which of the two states a launch settles in differs from chip to chip and from run to run (measured at
    // 32768 x 1536 x 1536: 53-57 us in step, 45-46 us out of step; with the late start always the latter).
    if (((int)blockIdx.x >> 3) & 1)
        for (int i = 0; i < late; ++i) __builtin_amdgcn_s_sleep(16);
    if constexpr (PAIR != 0) {
        if (!next_of_pair()) return;
    } else {
        plan_tile((int)blockIdx.x);
    }
    big4_issue_scales(plan, 0, 0);  // K >= 512: the first block is a whole one
    big4_issue_codes(plan, 0, 0);
    big4_issue_codes(plan, 1, 1);
    big4_issue_codes(plan, 2, 2);
    big4_issue_codes(plan, 3, 3);

    // scale block 0 and code stage 0 must be in; stages 1..3 (24 loads, the youngest) may be pending
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(24));
    __syncthreads();
    Big4State st;
    big4_read_scales(smem_bytes + kScaleAreaOff, a_sc_off, b_sc_off, st.sr);
    big_read_sub(smem_bytes, a_off0, b_off0, st.f0);

    int par = 0;
    stamp();
    [[maybe_unused]] bool more = true;
    for (int t = (int)blockIdx.x; PAIR ? more : t < total_items; t += stride) {
        v16f acc[4][4];
        const int64_t m0 = (int64_t)load_tm * kBigM, n0 = (int64_t)load_tn * kBigN;  // the load stream is still in item t
        const int cur_split = PAIR ? 0 : load_split;
        int rows = M, steps_real = nk_real;   // of the product that the tile belongs to
        int result = ROT ? BIG4_ROTATED : BIG4_PLAIN;
        [[maybe_unused]] RotEpilogue turn = rot;
        void* dst = c;
        if constexpr (PAIR != 0) {
            result = other.long_kind;
            if (load_short) {
                rows = other.M;
                steps_real = other.K / kBK;
                result = other.kind;
                turn = other.rot;
                dst = other.c;
            }
        }
        const int steps = PAIR ? (steps_real + 3) & ~3 : nk, muted_steps = PAIR ? steps - steps_real : muted;
        const int rows_valid = (int)(rows - m0) - wm * 128, cols_valid = (int)(N - n0) - wn * 128;
        // One block of four K steps.  The load stream is four K steps ahead and rolls over into the next tile;
        // after the last tile it re-requests the current steps (never consumed), which keeps the outstanding-load
        // counts uniform.  FIRST: the tile's first products overwrite the accumulators instead of adding to them.
        // the fused epilogue's mask words: one per 32 x 32 block of the lane's row, requested here -- ahead of the tile's
        // first K step, so that the K loop hides their latency -- into registers the epilogue reads.  A row's four words
        // (the wave's 128 columns) are 16 contiguous bytes: one request per block row.  A wave whose columns hang over the
        // edge of N by half requests the row's last 16 bytes (its own two words come second there); rows below M and
        // waves wholly outside read the matrix's last row / columns and store nothing.
        // Nothing may read these registers before the epilogue (the data is in flight): the words are picked there.
        [[maybe_unused]] u32x4 keep[4];
        [[maybe_unused]] bool keep_shifted = false;
        if constexpr (ROT) {
            // a plain product of a pair has no mask: its requests, which the counts of pending ones include, read 16 bytes of A
            const int64_t mask_pitch = PAIR && result == BIG4_PLAIN ? 0 : N / 8;
            int64_t ncol = n0 + wn * 128;
            keep_shifted = ncol + 128 > N;   // wave-uniform; N >= 256
            ncol = keep_shifted ? (int64_t)N - 128 : ncol;
            if (PAIR && result == BIG4_PLAIN) ncol = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                int64_t mrow = m0 + wm * 128 + i * 32 + lrow;
                mrow = mrow < rows ? mrow : (int64_t)rows - 1;
                const uint8_t* src = turn.mask + mrow * mask_pitch + ncol / 8;
                asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(keep[i]) : "v"(src) : "memory");
            }
        }
        auto block4 = [&](int ks, auto first) {
            constexpr bool FIRST = decltype(first)::value;
            // the four mask-word requests are younger than the stages the first block's steps 0..2 wait for
            constexpr int EX = (FIRST && ROT) ? 4 : 0;
            int lks = ks + 4;
            if (lks == steps) {
                if constexpr (PAIR != 0) {
                    more = next_of_pair();
                    lks = more ? 0 : ks;
                } else if (t + stride < total_items) {
                    plan_tile(t + stride);
                    lks = 0;
                } else {
                    lks = ks;
                }
            }
            const int lbase = lks + 4 <= steps_real ? lks : steps_real - 4;    // a short last block: the row's final four steps (a next tile's first: 0)
            const int first_live = ks + 4 > steps_real ? muted_steps : 0;      // this block's steps below it are muted
            const auto sw = [&](int q) { return q < first_live ? 0 : 16; };
            big4_step<0, sizeof(OutT) == 2, FIRST, EX>(plan, smem_bytes, lbase, lbase * 4, sw(0), par, a_off0, a_off1, b_off0, b_off1, a_sc_off, b_sc_off, sh, st, acc);
            big4_step<1, sizeof(OutT) == 2, false, EX>(plan, smem_bytes, lbase + 1, 0, sw(1), par, a_off0, a_off1, b_off0, b_off1, a_sc_off, b_sc_off, sh, st, acc);
            big4_step<2, sizeof(OutT) == 2, false, EX>(plan, smem_bytes, lbase + 2, 0, sw(2), par, a_off0, a_off1, b_off0, b_off1, a_sc_off, b_sc_off, sh, st, acc);
            big4_step<3, sizeof(OutT) == 2>(plan, smem_bytes, lbase + 3, 0, sw(3), par, a_off0, a_off1, b_off0, b_off1, a_sc_off, b_sc_off, sh, st, acc);
            par ^= 1;
        };
        block4(0, std::true_type{});
        for (int ks = 4; ks < steps; ks += 4) block4(ks, std::false_type{});
        stamp();
        if constexpr (PAIR != 0) {
            const auto leave = [&](auto rotated, auto wide) {
                big4_epilogue_bf16<decltype(rotated)::value ? ROT : 0, RAGGED, decltype(wide)::value>(acc, alpha, dst, m0, n0, N, wm, wn, wave, lane, smem_bytes,
                                                                                            rows_valid, cols_valid, turn, keep, keep_shifted);
            };
            if ((PAIR & BIG4_PLAIN) && result == BIG4_PLAIN) {
                // a use of the words that the tile requested, so that their registers stay theirs until they have arrived
#pragma unroll
                for (int i = 0; i < 4; ++i) asm volatile("" ::"v"(keep[i]));
                leave(std::false_type{}, std::false_type{});
            } else if ((PAIR & BIG4_WIDE) && ((PAIR & BIG4_ROTATED) == 0 || result == BIG4_WIDE)) leave(std::true_type{}, std::true_type{});
            else leave(std::true_type{}, std::false_type{});
        } else if constexpr (sizeof(OutT) == 2) {
            big4_epilogue_bf16<ROT, RAGGED, false, UNIT>(acc, alpha, dst, m0, n0, N, wm, wn, wave, lane, smem_bytes, rows_valid, cols_valid, turn, keep, keep_shifted);
        } else {
            OutT* slab = splits > 1 ? c + (int64_t)cur_split * M * N : c;
            const float a_eff = splits > 1 ? 1.0f : alpha;
            acc_settle();
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (i * 32 < rows_valid && j * 32 < cols_valid) {
                        const int64_t row0 = m0 + wm * 128 + i * 32, col = n0 + wn * 128 + j * 32 + lrow;
                        store_tile<OutT, true>(acc[i][j], a_eff, slab, row0, col, N, half, RAGGED ? rows_valid - i * 32 : 32);
                    }
        }
        stamp();
    }
    // direct-to-LDS loads must not outlive the workgroup's LDS allocation
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
}

// c[i] = alpha * (p[0][i] + p[1][i] + ... ) in slab order: the fixed order makes split-K results reproducible
template <typename OutT>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int splits, int64_t mn,
                                                            float alpha, OutT* __restrict__ c) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= mn) return;  // mn is a multiple of 4 (N % 64 == 0)
    float4 acc = *reinterpret_cast<const float4*>(partial + i);
    for (int s = 1; s < splits; ++s) {
        const float4 v = *reinterpret_cast<const float4*>(partial + (int64_t)s * mn + i);
        acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
    }
    acc.x *= alpha; acc.y *= alpha; acc.z *= alpha; acc.w *= alpha;
    if constexpr (sizeof(OutT) == 4) {
        *reinterpret_cast<float4*>(c + i) = acc;
    } else {
        const uint32_t lo = (uint32_t)f32_to_bf16(acc.x) | ((uint32_t)f32_to_bf16(acc.y) << 16);
        const uint32_t hi = (uint32_t)f32_to_bf16(acc.z) | ((uint32_t)f32_to_bf16(acc.w) << 16);
        *reinterpret_cast<uint2*>(c + i) = make_uint2(lo, hi);
    }
}

// Measurement aid: the block-scaled FP4 matrix instruction alone, on operand bytes taken from `operands`, with no
// memory traffic inside the loop.  What a wave of the GEMM does between its loads: 16 products per iteration on a 4 x 4
// grid of 32 x 32 accumulator blocks.  The rate this reaches on real operand bytes is the chip's ceiling for the
// product at its power limit (the clock it sustains depends on how much the operand bits toggle).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mfma_only_kernel(const uint4* __restrict__ operands,
                                                                                                    float* __restrict__ sink, int iters) {
    const int tid = threadIdx.x;
    uint4 a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        a[i] = operands[((size_t)blockIdx.x * 8 + i) * 256 + tid];
        b[i] = operands[((size_t)blockIdx.x * 8 + 4 + i) * 256 + tid];
    }
    v16f acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    const int sc = 0x7f7f7f7f;  // scale 2^0
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const v8i av = v8i{(int)a[i].x, (int)a[i].y, (int)a[i].z, (int)a[i].w, 0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const v8i bv = v8i{(int)b[j].x, (int)b[j].y, (int)b[j].z, (int)b[j].w, 0, 0, 0, 0};
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, acc[i][j], 4, 4, 0, sc, 0, sc);
            }
        }
    }
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) sum += acc[i][j][e];
    sink[(size_t)blockIdx.x * 256 + tid] = sum;
}

// ---- which kernel serves a product ----------------------------------------------------------------------------------
// Estimated durations in microseconds, fitted to 70 shapes of 0.2 to 740 GF with tiled operands: every kernel that serves the
// shape and cuts into 2 to 4 K ranges, each launch between two 8192 x 4096 x 4096 products (alone and back to back the kernels run at
// another clock and in another order of speed): mean error 6 %, and the choice costs 0.3 % more than the fastest on average.
// The 128 x 128 line is that of three stages: with one tile to a CU the kernel has a fourth (gemm_tile.hip) and is up to a fifth faster than it says.
// All kernels chosen from here give the same bits except a cut into K ranges, so nothing but time hangs on the choice.  (A
// layer's forward product of at most 64 tokens may run on gemm_rows.hip instead, before this choice; its sums are in another
// order.)
struct KernelCost {
    int bm, bn, per_cu;              // tile, resident workgroups per CU
    double step, shared, boundary;   // one K step of a workgroup alone on its CU; with n of them: n * shared; per tile
    double rotate[3], more[3];       // what the rotation (blocks of 32, 64, 128) adds to the first round of per_cu tiles and to each further one
};
constexpr KernelCost kTileCosts[] = {{256, 128, 2, 0.461, 0.488, 5.6, {5.8, 6.2, 12.0}, {8.0, 9.0, 11.0}},
                                     {128, 128, 3, 0.155, 0.294, 1.71, {3.2, 3.7, 4.5}, {1.9, 2.4, 4.0}},
                                     {128, 64, 3, 0.172, 0.204, 0.99, {1.6, 2.9, 0.0}, {1.2, 1.5, 0.0}},
                                     {64, 64, 4, 0.152, 0.129, 0.72, {0.6, 1.6, 0.0}, {0.75, 1.2, 0.0}},
                                     {64, 32, 4, 0.099, 0.091, 0.71, {0.7, 0.0, 0.0}, {0.7, 0.0, 0.0}}};
// 256 x 128 tiles over fewer than kShortTallSteps K steps, which request their scales step by step
constexpr KernelCost kShortTall = {256, 128, 2, 0.60, 0.68, 2.5, {5.8, 6.2, 12.0}, {8.0, 9.0, 11.0}};
// with a B of six or eight bits (expand.hip; fitted to six bits in 14 shapes of 512 x 640 x 2048 to 4096^3, rotation included)
constexpr KernelCost kWideTileCosts[] = {{256, 256, 1, 1.14, 1.14, 4.0, {9.0, 10.9, 12.3}, {10.0, 11.0, 12.3}},
                                         {128, 128, 3, 0.45, 0.33, 3.0, {7.0, 7.2, 8.0}, {2.0, 2.4, 4.0}},
                                         {128, 64, 3, 0.31, 0.24, 1.0, {2.4, 3.6, 0.0}, {0.8, 2.2, 0.0}},
                                         {64, 64, 3, 0.21, 0.18, 0.60, {1.0, 1.5, 0.0}, {0.8, 1.4, 0.0}}};
const KernelCost& tile_costs(bool e5m2, int kind, int64_t K, int splits) {
    if (!e5m2 && kind == TILE_256x128 && K / kBK / splits < kShortTallSteps) return kShortTall;
    return (e5m2 ? kWideTileCosts : kTileCosts)[kind];
}
int last_tile_kind(bool e5m2) { return e5m2 ? TILE_64x64 : TILE_64x32; }
constexpr double kLaunch = 3.0, kPersistentStep = 0.675, kPersistentBoundary = 5.5, kPersistentMuted = 1.6;
double persistent_rotate_cost(int hd) { return hd == 32 ? 3.9 : hd == 64 ? 4.5 : 5.0; }
constexpr double kMemory = 5.5e6, kRotateMemory = 5.2e6, kWideStores = 1.0e7;   // bytes per us of the reduction, of a rotation pass of its own, of what fp32 results add

double ranges_cost(int64_t M, int64_t N, int splits) {   // writing, reading and reducing the partial sums of a cut product
    return splits == 1 ? 0.0 : kLaunch + (4.0 * splits + 2.0) * (double)M * (double)N / kMemory;
}
double tile_cost(const KernelCost& k, int64_t M, int64_t N, int64_t K, int splits, int cus) {
    const int64_t tiles = ((M + k.bm - 1) / k.bm) * ((N + k.bn - 1) / k.bn) * splits, all = (K + kBK - 1) / kBK, steps = (all + splits - 1) / splits;
    const auto round = [&](int64_t n) {   // n workgroups of one CU side by side
        const double step = k.step > n * k.shared ? k.step : n * k.shared;
        return steps * step + k.boundary * __builtin_sqrt((double)n);
    };
    const int64_t full = tiles / (k.per_cu * cus), rest = tiles % (k.per_cu * cus);
    return kLaunch + full * round(k.per_cu) + (rest ? round((rest + cus - 1) / cus) : 0.0) + ranges_cost(M, N, splits);
}
// 256 x 192 tiles, two to a CU (gemm_two.hip).  Fewer than one a CU leave it to a workgroup that nothing covers; with one on some CUs and two on
// others the chip runs them faster than with two everywhere.  Fitted to 106 shapes of 0.6 to 370 GF with tiled operands, each launch behind a copy of
// 32 MiB: rms error 7 %.  Taken where it is below kTwoMargin of the cheapest other kernel, which costs 0.25 % more than the fastest
// on average and is slower than it by 2 % and more in two of the shapes.  us, the other kernel and this one: 16384 x 1536 x 4096 57.2 and 52.5, 13328 x
// 1280 x 2176 28.8 and 26.7, 16832 x 9280 x 2176 204.5 and 179.8, 26256 x 4672 x 768 84.6 and 74.1; where the line lies 17152 x 5184 x 1792 92.5 and 95.3,
// 9120 x 9600 x 1920 99.0 and 99.3; left to the others 8192 x 4096^2 65.4 and 75.4, 4096^3 34.8 and 43.4.
constexpr double kTwoMargin = 0.95;
double two_cost(int64_t M, int64_t N, int64_t K, int cus) {
    const int64_t tiles = ((M + 255) / 256) * ((N + 191) / 192), steps = K / kBK, full = tiles / (2 * cus), rest = tiles % (2 * cus);
    if (tiles <= cus) return 1e30;
    const double both = 1.3, one = 0.78, some = 1.1, boundary = 5.5;
    double cost = kLaunch + 1.0 + full * (steps * both + boundary);
    if (rest > cus) cost += steps * (some + (both - some) * (double)(rest - cus) / cus) + boundary;
    else if (rest) cost += steps * one + 3.15;
    return cost;
}
// the masked inverse rotation in the epilogue of a tile kernel, and as a kernel of its own
double tile_rotate_cost(const KernelCost& k, int64_t M, int64_t N, int hd, int out_bytes, int cus) {
    const int64_t tiles = ((M + k.bm - 1) / k.bm) * ((N + k.bn - 1) / k.bn);
    const double rounds = (double)((tiles + cus - 1) / cus) / k.per_cu;
    const int h = hd == 32 ? 0 : hd == 64 ? 1 : 2;
    return k.rotate[h] + (rounds > 1.0 ? (rounds - 1.0) * k.more[h] : 0.0) + (double)M * (double)N * (out_bytes - 2) / kWideStores;
}
double separate_rotate_cost(int64_t M, int64_t N, int in_bytes, int out_bytes) {
    return kLaunch + 0.5 + (double)M * (double)N * (in_bytes + out_bytes) / kRotateMemory;
}
double persistent_cost(int64_t M, int64_t N, int64_t K, int splits, int cus) {
    const int64_t items = ((M + kBigM - 1) / kBigM) * ((N + kBigN - 1) / kBigN) * splits;
    const int64_t steps = (K / kBK / splits + 3) & ~(int64_t)3;
    const double boundary = kPersistentBoundary + (K % 512 ? kPersistentMuted : 0.0);
    return kLaunch + (double)((items + cus - 1) / cus) * (steps * kPersistentStep + boundary) + ranges_cost(M, N, splits);
}

// The persistent kernel: M any, N a multiple of 64, at least one tile; it walks K in blocks of four steps: K % 512 == 0
// directly (scale rows are then 16-byte aligned like their base), other multiples of 128 with up to three muted steps in
// the last block; their 16-byte scale requests start at 4-byte aligned addresses.  Not five steps: with three of eight muted the
// tile kernels are cheaper for every M and N, with the rotation and without.  Muted steps cost what others do, and their
// tile 1.6 us more at its boundary, and the estimate counts them (16480 x 1728 x 640 with the rotation: 33 us, 28 on 128 x 128
// tiles).  (Passing over the products of a muted step instead, by a branch, makes the compiler keep a second set of
// accumulators, in memory.)
bool persistent_serves(int64_t M, int64_t N, int64_t K, const void* a_scales, const void* b_scales, const void* c) {
    const int64_t steps = K / kBK;
    if (N % 64 || M < kBigM || N < kBigN || K % kBK || steps < 4 || steps == 5 || M >= (1 << 30) || N >= (1 << 30) || K >= (1 << 26)) return false;
    if (K % 512 == 0 && ((reinterpret_cast<uintptr_t>(a_scales) | reinterpret_cast<uintptr_t>(b_scales)) & 15)) return false;
    return (reinterpret_cast<uintptr_t>(c) & 15) == 0;
}

// The rotation in the persistent kernel's epilogue: column signs that are the same in every 32 of a block of 64 or 128 (none, in a
// layer whose forward quantizers are not re-randomized)
bool persistent_rotates(const TileProduct& p) {
    for (int j = 1; j < p.hd / 32; ++j)
        if (p.signs.w[j] != p.signs.w[0]) return false;
    return p.N % p.hd == 0;
}

// The cheapest cut of a product into K ranges (splits == 1: none is possible): each range keeps at least four K steps, on the
// persistent kernel whole blocks of four steps and at least two of them.  Few tiles and a long K leave CUs idle: 640 x 1728 x
// 16512 took 49 us whole and 32 us in three ranges of 128 x 128 tiles, 1536 x 4096 x 16384 110 us and 71 us in two ranges.
struct Cut {
    ProductChoice choice;
    double cost;
};
Cut cheapest_cut(int64_t M, int64_t N, int64_t K, bool persistent, bool tiles_ok, bool e5m2, int cus) {
    Cut best{{ProductChoice::GENERIC, 0, 1, false}, 1e30};
    const int64_t steps = (K + kBK - 1) / kBK;
    const auto consider = [&](ProductChoice::Path path, int kind, int sp, double cost) {
        if (cost < best.cost) best = Cut{{path, kind, sp, false}, cost};
    };
    for (int sp = 2; sp <= 32 && steps / sp >= 4; ++sp) {
        if (persistent && K % 512 == 0 && (K / 512) % sp == 0 && K / 512 / sp >= 2)
            consider(ProductChoice::PERSISTENT, 0, sp, persistent_cost(M, N, K, sp, cus));
        if (tiles_ok)
            for (int kind = TILE_256x128; kind <= TILE_64x64; ++kind) consider(ProductChoice::TILE, kind, sp, tile_cost(tile_costs(e5m2, kind, K, sp), M, N, K, sp, cus));
    }
    return best;
}

// late start (units of 1024 cycles) of every other group of workgroups: contractions of at most sixteen K steps per work
// item, where the tile boundary is a third or more of a tile; longer ones neither gain nor lose (within 0.7 %)
int big4_late_start(int64_t K, int splits) { return K / kBK / splits <= 16 ? 6 : 0; }

template <typename OutT, int ROT, bool RAGGED, bool UNIT = false>
hipError_t launch_big4_as(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                          const uint8_t* b_scales, int64_t M, int64_t N, int64_t K, float alpha, void* c, int a_tiled,
                          int b_tiled, int splits, int cus, hipStream_t stream, const RotEpilogue& rot) {
    auto kern = gemm_mxfp4_tn_big4_kernel<OutT, false, ROT, RAGGED, 0, UNIT>;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    hipError_t e = allow_dynamic_lds(kern, kBig4SmemBytes, lds_allowed);
    if (e != hipSuccess) return e;
    const int64_t items = ((M + kBigM - 1) / kBigM) * ((N + kBigN - 1) / kBigN) * splits;
    // one workgroup per CU, and where a workgroup walks several items a grid that is a multiple of 8, so that item t and
    // t + grid land on the same XCD
    int64_t g = items < cus ? items : cus;
    if (g > 8 && g < items) g -= g % 8;
    dim3 grid((unsigned)g), block(256);
    kern<<<grid, block, kBig4SmemBytes, stream>>>(a_codes, a_scales, b_codes, b_scales, (int)M, (int)N, (int)K, alpha,
                                                  reinterpret_cast<OutT*>(c), a_tiled, b_tiled, splits, big4_late_start(K, splits), nullptr, rot, Big4NoOther{});
    return hipGetLastError();
}
template <typename OutT, int ROT = 0>
hipError_t launch_big4(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                       const uint8_t* b_scales, int64_t M, int64_t N, int64_t K, float alpha, void* c, int a_tiled,
                       int b_tiled, int splits, int cus, hipStream_t stream, const RotEpilogue& rot = RotEpilogue{}) {
    if constexpr (sizeof(OutT) == 2 && ROT == 0)
        if (alpha == 1.0f)
            return M % 64 ? launch_big4_as<OutT, 0, true, true>(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, a_tiled, b_tiled, splits, cus, stream, rot)
                          : launch_big4_as<OutT, 0, false, true>(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, a_tiled, b_tiled, splits, cus, stream, rot);
    if (M % 64)
        return launch_big4_as<OutT, ROT, true>(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, a_tiled, b_tiled, splits, cus, stream, rot);
    return launch_big4_as<OutT, ROT, false>(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, a_tiled, b_tiled, splits, cus, stream, rot);
}

template <int BM, int BN, int WM, int WN>
hipError_t launch_gemm(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                       const uint8_t* b_scales, int64_t M, int64_t N, int64_t K, float alpha, void* c, int c_dtype,
                       hipStream_t stream) {
    dim3 grid((unsigned)((N + BN - 1) / BN), (unsigned)((M + BM - 1) / BM)), block(256);
    constexpr int smem = GemmSmem<BM, BN>::kBytes;
    if (c_dtype == BF16) {
        auto kern = gemm_mxfp4_tn_kernel<BM, BN, WM, WN, uint16_t>;
        if (smem > 48 * 1024) {
            static std::atomic<bool> lds_allowed[kMaxDevices];
            hipError_t e = allow_dynamic_lds(kern, smem, lds_allowed);
            if (e != hipSuccess) return e;
        }
        kern<<<grid, block, smem, stream>>>(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, reinterpret_cast<uint16_t*>(c));
    } else {
        auto kern = gemm_mxfp4_tn_kernel<BM, BN, WM, WN, float>;
        if (smem > 48 * 1024) {
            static std::atomic<bool> lds_allowed[kMaxDevices];
            hipError_t e = allow_dynamic_lds(kern, smem, lds_allowed);
            if (e != hipSuccess) return e;
        }
        kern<<<grid, block, smem, stream>>>(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, reinterpret_cast<float*>(c));
    }
    return hipGetLastError();
}

}  // namespace

// one launch of the persistent kernel's stamping instantiation (bf16 output, no K ranges); returns its grid size, 0 on
// shapes that kernel does not serve.  stamps: device memory for grid * kPhaseStamps 64-bit values.
int gemm_phase_stamps_per_group() { return kPhaseStamps; }
hipError_t gemm_tile_phases(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales,
                            int64_t M, int64_t N, int64_t K, float alpha, void* c, int a_layout, int b_layout,
                            const uint8_t* rot_mask, unsigned long long* stamps, size_t stamps_bytes, int* grid_out, hipStream_t stream) {
    *grid_out = 0;
    if (!gemm_supports_tiled(M, N, K) || K % 512 || ((reinterpret_cast<uintptr_t>(a_scales) | reinterpret_cast<uintptr_t>(b_scales)) & 15))
        return hipErrorInvalidValue;
    // rot_mask: the instantiation whose epilogue carries the masked inverse rotation (no sign flips, bf16 scale)
    auto kern = rot_mask ? gemm_mxfp4_tn_big4_kernel<uint16_t, true, 32> : gemm_mxfp4_tn_big4_kernel<uint16_t, true, 0>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kBig4SmemBytes);
    if (e != hipSuccess) return e;
    const int64_t items = ((M + kBigM - 1) / kBigM) * ((N + kBigN - 1) / kBigN);
    const int cus = device_cus();
    int64_t g = items < cus ? items : cus;
    if (g > 8) g -= g % 8;
    if (stamps_bytes < (size_t)g * kPhaseStamps * sizeof(unsigned long long)) return hipErrorInvalidValue;
    kern<<<dim3((unsigned)g), dim3(256), kBig4SmemBytes, stream>>>(a_codes, a_scales, b_codes, b_scales, (int)M, (int)N, (int)K, alpha,
                                                                  reinterpret_cast<uint16_t*>(c), a_layout == LAYOUT_TILED,
                                                                  b_layout == LAYOUT_TILED, 1, big4_late_start(K, 1), stamps,
                                                                  RotEpilogue{rot_mask, 0u, hadamard_scale(32, BF16)}, Big4NoOther{});
    *grid_out = (int)g;
    return hipGetLastError();
}

// one workgroup (four waves, one per SIMD) per CU; reads blocks * 32 KiB of operands, writes blocks * 256 floats
int mfma_only_blocks() { return device_cus(); }
hipError_t mfma_only(const uint8_t* operands, float* sink, int iters, hipStream_t stream) {
    mfma_only_kernel<<<dim3((unsigned)device_cus()), dim3(256), 0, stream>>>(reinterpret_cast<const uint4*>(operands), sink, iters);
    return hipGetLastError();
}

// Shapes the 256x256-tile kernels serve (they also read tiled operands): extents multiples of 64 and at least one
// full tile wide, K a multiple of 128; tiles hanging over the edge of M or N compute on clamped rows and store nothing there.
bool gemm_supports_tiled(int64_t M, int64_t N, int64_t K) {
    return M % 64 == 0 && N % 64 == 0 && M >= kBigM && N >= kBigN && K > 0 && K % kBK == 0 && M < (1 << 30) && N < (1 << 30) &&
           K < (1 << 30);
}

// The candidates of one shape, worked out once per thread and remembered (a layer's backward pass asks for two or more shapes
// several times over; 160 estimates take the host up to several microseconds): up to 256 shapes, 40 KB
struct ShapePlan {
    int64_t M = -1, N = 0, K = 0;
    int flags = -1;
    double persistent = 1e30, two = 1e30, tile[5] = {};
    Cut cut{};
    size_t cut_bytes = 0;       // scratch of the cut, 0 if it would not be made
    size_t scratch_bytes = 0;   // what a caller is asked to provide: at least cut_bytes
};
// Few tiles of the persistent kernel and a long K: callers hold room for its ranges that would fill the CUs, whether or not a cut
// turns out cheaper than the whole product (it mostly does from 64 K steps on).
size_t scratch_of_few_tiles(int64_t M, int64_t N, int64_t K, int cus) {
    const int64_t tiles = ((M + kBigM - 1) / kBigM) * ((N + kBigN - 1) / kBigN), nblk = K / 512;
    if (K % 512 || tiles * 4 >= cus * 3 || nblk < 4) return 0;
    double best = 1e30;
    int splits = 1;
    for (int sp = 1; sp <= nblk && sp <= 64; ++sp) {
        if (nblk % sp || (nblk / sp) * 4 < 8) continue;
        const double cost = (double)((tiles * sp + cus - 1) / cus) * ((double)(nblk / sp) * 4 + 6.0) + (sp > 1 ? 4.0 + 0.5 * sp : 0.0);
        if (cost < best - 1e-9) {
            best = cost;
            splits = sp;
        }
    }
    return splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
}
ShapePlan make_plan(int64_t M, int64_t N, int64_t K, bool persistent, bool tiles_ok, bool e5m2, int flags) {
    const int cus = device_cus();
    ShapePlan p;
    p.M = M; p.N = N; p.K = K; p.flags = flags;
    double best = 1e30;
    if (persistent) best = p.persistent = persistent_cost(M, N, K, 1, cus);
    p.two = two_cost(M, N, K, cus);
    for (int kind = TILE_256x128; kind <= last_tile_kind(e5m2); ++kind) {
        p.tile[kind] = tiles_ok ? tile_cost(tile_costs(e5m2, kind, K, 1), M, N, K, 1, cus) : 1e30;
        best = p.tile[kind] < best ? p.tile[kind] : best;
    }
    p.cut = cheapest_cut(M, N, K, persistent, tiles_ok, e5m2, cus);
    p.cut_bytes = p.cut.cost < best ? (size_t)p.cut.choice.splits * (size_t)M * (size_t)N * sizeof(float) : 0;
    p.scratch_bytes = persistent ? scratch_of_few_tiles(M, N, K, cus) : 0;
    if (p.cut_bytes > p.scratch_bytes) p.scratch_bytes = p.cut_bytes;
    return p;
}
const ShapePlan& plan_of_shape(int64_t M, int64_t N, int64_t K, bool persistent, bool tiles_ok, bool e5m2 = false) {
    static thread_local ShapeTable<ShapePlan, 6> table;
    const int flags = (persistent ? 1 : 0) | (tiles_ok ? 2 : 0) | (e5m2 ? 4 : 0);
    return table.find(M, N, K, flags, [&] { return make_plan(M, N, K, persistent, tiles_ok, e5m2, flags); });
}

// bytes of scratch with which gemm_mxfp4_tn makes every cut into K ranges that it would make of this shape (0: it would make none;
// scratch_of_few_tiles asks for some that may go unused)
size_t gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    const bool persistent = persistent_serves(M, N, K, nullptr, nullptr, nullptr), tiles_ok = gemm_tile_serves(M, N, K, 0, 0, nullptr);
    return persistent || tiles_ok ? plan_of_shape(M, N, K, persistent, tiles_ok).scratch_bytes : 0;
}
size_t gemm_few_tiles_bytes(int64_t M, int64_t N, int64_t K) { return gemm_supports_tiled(M, N, K) ? scratch_of_few_tiles(M, N, K, device_cus()) : 0; }
size_t gemm_e5m2_workspace_bytes(int64_t M, int64_t N, int64_t K) { return plan_of_shape(M, N, K, false, true, true).scratch_bytes; }

// The kernel that serves product p.  p.mask: the caller wants the masked inverse rotation applied to the result (mid dtype
// c_dtype, stored in rot_out_dtype); `rotates` tells whether the chosen kernel does it.  Where it does not, the rotation is
// a kernel of its own that reads and writes the result, which the comparison accounts for.
ProductChoice choose_product(const TileProduct& p, int c_dtype, int rot_out_dtype, const void* workspace, size_t workspace_bytes) {
    const int64_t M = p.M, N = p.N, K = p.K;
    const bool rotate = p.mask != nullptr;
    const bool e5m2 = p.b_e5m2;
    const bool persistent = !e5m2 && persistent_serves(M, N, K, p.a_scales, p.b_scales, p.c);
    const bool tiles_ok = gemm_tile_serves(M, N, K, p.a_tiled, p.b_tiled, p.c);
    if (!persistent && !tiles_ok) return {ProductChoice::GENERIC, 0, 1, false};
    const ShapePlan& plan = plan_of_shape(M, N, K, persistent, tiles_ok, e5m2);
    // a cut into K ranges rounds differently: whether to make it is decided on the product alone, so that a product and the
    // same product with the rotation agree (a layer's two gradients may share a launch instead, without cuts: see gradient_pair)
    if (plan.cut_bytes && workspace && plan.cut_bytes <= workspace_bytes && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0) {
        ProductChoice c = plan.cut.choice;
        c.rotates = rotate;
        c.cost = plan.cut.cost;
        return c;
    }
    const double separate = rotate ? separate_rotate_cost(M, N, c_dtype == BF16 ? 2 : 4, rot_out_dtype == BF16 ? 2 : 4) : 0.0;
    ProductChoice best{ProductChoice::GENERIC, 0, 1, false};
    double best_cost = 1e30;
    const auto consider = [&](ProductChoice c, double cost) {
        if (cost < best_cost) {
            best_cost = cost;
            best = c;
            best.cost = cost;
        }
    };
    const bool bf16 = c_dtype == BF16;
    const int cus = device_cus();
    if (persistent) {
        if (rotate && bf16 && rot_out_dtype == BF16 && persistent_rotates(p)) consider({ProductChoice::PERSISTENT, 0, 1, true}, plan.persistent + persistent_rotate_cost(p.hd));
        consider({ProductChoice::PERSISTENT, 0, 1, false}, plan.persistent + separate);
    }
    for (int kind = TILE_256x128; tiles_ok && kind <= last_tile_kind(e5m2); ++kind) {
        const KernelCost& k = tile_costs(e5m2, kind, K, 1);
        if (rotate && bf16 && k.bn >= p.hd) consider({ProductChoice::TILE, kind, 1, true}, plan.tile[kind] + tile_rotate_cost(k, M, N, p.hd, rot_out_dtype == BF16 ? 2 : 4, cus));
        consider({ProductChoice::TILE, kind, 1, false}, plan.tile[kind] + separate);
    }
    if (!rotate && bf16 && plan.two < kTwoMargin * best_cost && gemm_two_serves(p)) consider({ProductChoice::TWO, 0, 1, false}, plan.two);
    return best;
}

// Runs product p on the chosen kernel.  Rotated (c.rotates): p.c receives rot_out_dtype elements; otherwise the plain product
// in c_dtype.  workspace as offered to choose_product.
hipError_t run_product(const ProductChoice& c, const TileProduct& p, int c_dtype, int rot_out_dtype, void* workspace, hipStream_t stream) {
    const int64_t M = p.M, N = p.N, K = p.K;
    const int cus = device_cus();
    if (c.path == ProductChoice::GENERIC) {
        if (p.a_tiled || p.b_tiled || p.b_e5m2) return hipErrorInvalidValue;
        return launch_gemm<128, 128, 64, 64>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, M, N, K, p.alpha, p.c, c_dtype, stream);
    }
    if (c.splits > 1) {
        // partial sums per K range in fp32 (plain accumulator layout), then one ordered reduction
        hipError_t e;
        if (c.path == ProductChoice::TILE) {
            TileProduct q = p;
            q.c = workspace;
            q.splits = c.splits;
            q.mask = nullptr;
            e = gemm_tile(c.kind, q, F32, stream);
        } else {
            e = launch_big4<float>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, M, N, K, 1.0f, workspace, p.a_tiled, p.b_tiled, c.splits, cus, stream);
        }
        if (e != hipSuccess) return e;
        const int64_t mn = M * N;
        const float* part = static_cast<const float*>(workspace);
        if (c.rotates)
            return splitk_reduce_rotated(part, c.splits, mn, p.alpha, c_dtype, p.mask, p.hd, p.signs, p.rot_c, p.c, rot_out_dtype, stream);
        dim3 grid((unsigned)((mn / 4 + 255) / 256)), block(256);
        if (c_dtype == BF16)
            splitk_reduce_kernel<uint16_t><<<grid, block, 0, stream>>>(part, c.splits, mn, p.alpha, static_cast<uint16_t*>(p.c));
        else
            splitk_reduce_kernel<float><<<grid, block, 0, stream>>>(part, c.splits, mn, p.alpha, static_cast<float*>(p.c));
        return hipGetLastError();
    }
    if (c.path == ProductChoice::TWO) return c_dtype == BF16 ? gemm_two(p, stream) : hipErrorInvalidValue;
    if (c.path == ProductChoice::TILE) {
        TileProduct q = p;
        q.splits = 1;
        if (!c.rotates) q.mask = nullptr;
        q.out_f32 = c_dtype == BF16 && rot_out_dtype == F32;
        return gemm_tile(c.kind, q, c_dtype, stream);
    }
    if (c.rotates) {
        const auto rotated = [&](auto hd) {
            return launch_big4<uint16_t, decltype(hd)::value>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, M, N, K, p.alpha, p.c, p.a_tiled, p.b_tiled, 1, cus, stream,
                                                              RotEpilogue{p.mask, p.signs.w[0], p.rot_c});
        };
        return p.hd == 32 ? rotated(std::integral_constant<int, 32>{}) : p.hd == 64 ? rotated(std::integral_constant<int, 64>{}) : rotated(std::integral_constant<int, 128>{});
    }
    if (c_dtype == BF16)
        return launch_big4<uint16_t>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, M, N, K, p.alpha, p.c, p.a_tiled, p.b_tiled, 1, cus, stream);
    return launch_big4<float>(p.a_codes, p.a_scales, p.b_codes, p.b_scales, M, N, K, p.alpha, p.c, p.a_tiled, p.b_tiled, 1, cus, stream);
}

// ---- the two gradient products of a layer in one launch --------------------------------------------------------------
namespace {
int64_t big_tiles(const TileProduct& p) { return (int64_t)((p.M + kBigM - 1) / kBigM) * ((p.N + kBigN - 1) / kBigN); }
int pair_grid(int64_t tiles, int cus) { return (int)(tiles < cus ? tiles : cus) & ~7; }   // as many workgroups on every XCD
double pair_tile_cost(int64_t K) { return ((K / kBK + 3) & ~(int64_t)3) * kPersistentStep + kPersistentBoundary + (K % 512 ? kPersistentMuted : 0.0); }
// when the last workgroup of the fullest XCD ends, and how many short tiles every workgroup takes first (see Big4Other)
double pair_makespan(const TileProduct& lng, const TileProduct& sht, int cus, int* rounds) {
    const int64_t tl = big_tiles(lng), ts = big_tiles(sht), W = pair_grid(tl + ts, cus) / 8, L = (tl + 7) / 8, S = (ts + 7) / 8, heavy = L % W;
    const double cl = pair_tile_cost(lng.K), cs = pair_tile_cost(sht.K);
    double best = 1e30;
    for (int64_t b = 0; b <= (S + W - 1) / W; ++b) {
        const int64_t left = S - W * b > 0 ? S - W * b : 0;
        const double all = (double)(L / W) * cl + b * cs, with = heavy ? all + cl : 0.0, without = all + (double)((left + W - heavy - 1) / (W - heavy)) * cs;
        const double end = with > without ? with : without;
        if (end < best) {
            best = end;
            *rounds = (int)b;
        }
    }
    return best;
}
template <int PAIR, int ROT, bool RAGGED>
hipError_t launch_pair_as(const TileProduct& lng, const Big4Other& other, const RotEpilogue& rot, int late, int grid, hipStream_t stream) {
    auto kern = gemm_mxfp4_tn_big4_kernel<uint16_t, false, ROT, RAGGED, PAIR>;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    const hipError_t e = allow_dynamic_lds(kern, kBig4SmemBytes, lds_allowed);
    if (e != hipSuccess) return e;
    kern<<<dim3((unsigned)grid), dim3(256), kBig4SmemBytes, stream>>>(lng.a_codes, lng.a_scales, lng.b_codes, lng.b_scales, lng.M, lng.N, lng.K, lng.alpha,
                                                                      static_cast<uint16_t*>(lng.c), 1, 1, 1, late, nullptr, rot, other);
    return hipGetLastError();
}
}  // namespace

// Served: both products by the persistent kernel, tiled, with at least one tile per CU between them (fewer leave CUs idle, which
// smaller tiles and K ranges do not) and eight K steps a tile (with four the larger product is bound by its stores, 541 MB of them in
// 24576 x 11008 x 512, which long tiles beside it leave to fewer CUs: 666 us, 632 in two launches); bf16 results, plain or with the rotation
// (both over the same block; beside a plain one over 32), one of them with it, and only rotated ones widened.  What is gained is the idle part
// of each product's last round, or writing and reading partial sums.  Worth it where the estimate of the one launch is below this part
// of the sum of the two products' own; whole training steps, two launches against one:
//   both on this kernel apart, too: one estimate on both sides.  8192 x 4096^2 (0.94) 294 -> 289, 16384 x 4096^2 and 4096 x 8192^2 (0.97)
//   545 -> 541 and 518 -> 517; of ten shapes from 0.94 to 0.98 one is slower, by 1.2 %.
constexpr double kPairLike = 0.97;
//   one of them cut into K ranges: 16384 x 1728 x 4096 (0.90) 333 -> 311, 32768 x 2048 x 3072 (0.91) 509 -> 502, 24576 x 1152 x 4608 (0.93)
//   410 -> 400; from 0.936 to 0.956 as many are slower (24576 x 6144 x 1152 with an fp32 weight 533 -> 553) as are faster (24576 x 1920 x 3456 437 -> 414).
constexpr double kPairCut = 0.935;
//   one of them whole on the tile kernels: 16480 x 3456 x 2048 (0.80) 342 -> 307, 12288 x 7168 x 1152 (0.87) 315 -> 300; 8192 x 7168 x 1152
//   (0.89) is even (219 -> 221 on one card, 221 -> 217 on another), 4096 x 2048 x 5504 (0.90) 141.5 -> 143.5, 4096 x 4096 x 4608 (0.94) 203 -> 213.
constexpr double kPairUnlike = 0.89;
double pair_margin(const ProductChoice& cx, const ProductChoice& cw) {
    if (cx.splits > 1 || cw.splits > 1) return kPairCut;
    return cx.path == ProductChoice::PERSISTENT && cw.path == ProductChoice::PERSISTENT ? kPairLike : kPairUnlike;
}
bool persistent_pair_serves(const TileProduct& x, int x_out, const TileProduct& w, int w_out) {
    const auto serves = [](const TileProduct& p, int out) {
        return p.a_tiled && p.b_tiled && (p.mask ? persistent_rotates(p) : out == BF16) && persistent_serves(p.M, p.N, p.K, p.a_scales, p.b_scales, p.c);
    };
    const int hd = x.mask ? x.hd : w.hd, cus = device_cus();
    return serves(x, x_out) && serves(w, w_out) && (x.mask && w.mask ? x.hd == w.hd : hd == 32) && cus >= 8 && big_tiles(x) + big_tiles(w) >= cus &&
           x.K >= 8 * kBK && w.K >= 8 * kBK;
}
double persistent_pair_cost(const TileProduct& x, int x_out, const TileProduct& w, int w_out, int cus) {
    int rounds;
    const bool x_long = x.K > w.K;
    double cost = kLaunch + pair_makespan(x_long ? x : w, x_long ? w : x, cus, &rounds) + persistent_rotate_cost(x.mask ? x.hd : w.hd);
    if (x.mask && x_out != BF16) cost += (double)x.M * x.N * 2 / kWideStores;
    if (w.mask && w_out != BF16) cost += (double)w.M * w.N * 2 / kWideStores;
    return cost;
}
// What a tile costs its CU among others of a pair, in us: a K step, the boundary, the rotation; and a K step of a tile whose CU has
// others beside it, of up to 12 steps (in their boundaries for a third of their time and more) and of more, and when they are done; its
// half of the launch, first fill and drain.  Fitted to 20 shapes from 512 x 640 x 1920 to 32768 x 1536 x 1536; the fifth figure to weight gradients of
// 192 and 256 steps beside tiles of 27 and 32: 32768 x 640 x 3456 and 24576 x 640 x 4096, which take 332 and 368 us a step in two launches
// (the gradient in three K ranges), 338 and 374 in one.
struct PairTile {
    int kind, bm;   // as many columns as rows
    double step, boundary, rotate, beside, beside_long, after, launch;
};
constexpr int kShortPairSteps = 12;
constexpr PairTile kPairTiles[] = {{TILE_128x128, 128, 0.26, 0.99, 0.63, 0.37, 0.45, 0.25, 3.5}, {TILE_64x64, 64, 0.129, 0.36, 0.19, 0.30, 0.30, 0.14, 2.0}};
// 60 other shapes: GPU time of the backward pass 0.92 of two launches' on average.  19 more from 0.80 to 0.90: whole steps 1.02 to 1.14 times as
// fast (16480 x 1728 x 640 122 -> 114.5, 24576 x 4608 x 640 324 -> 296); where gx is left rotated for the kernel behind it, 0.99 to 1.09
constexpr double kTilePairMargin = 0.9;
// Tiles go to the CUs as they become free, the longer contraction's first: every CU its share of those, then the others to even it
// out.  A tile of very many steps is still running when the others are done.
double tile_pair_cost(const TileProduct& x, int x_out, const PairTile& kx, const TileProduct& w, int w_out, const PairTile& kw, int cus) {
    const auto tiles = [](const TileProduct& p, const PairTile& k) { return (int64_t)((p.M + k.bm - 1) / k.bm) * ((p.N + k.bm - 1) / k.bm); };
    const auto tile = [](const TileProduct& p, const PairTile& k) { return p.K / kBK * k.step + k.boundary + (p.mask ? k.rotate : 0.0); };
    const bool x_long = x.K > w.K;
    const TileProduct &lng = x_long ? x : w, &sht = x_long ? w : x;
    const PairTile &kl = x_long ? kx : kw, &ks = x_long ? kw : kx;
    const int64_t tl = tiles(lng, kl), ts = tiles(sht, ks);
    const double cl = tile(lng, kl), cs = tile(sht, ks), mean = (tl * cl + ts * cs) / cus;
    const double most_long = (double)((tl + cus - 1) / cus) * cl;
    // the CUs with most of the long ones, and whole short ones up to the mean on the others
    const double even = mean + (ts > 0 ? 0.5 * cs : 0.0);
    double all = most_long > even ? most_long : even;
    if (tl % cus == 0) all = (double)(tl / cus) * cl + (double)((ts + cus - 1) / cus) * cs;
    const double left = lng.K / kBK - all / (sht.K / kBK <= kShortPairSteps ? kl.beside : kl.beside_long);
    double cost = kx.launch + kw.launch + all + (left > 0.0 ? left * kl.after : 0.0);
    if (x.mask && x_out != BF16) cost += (double)x.M * x.N * 2 / kWideStores;
    if (w.mask && w_out != BF16) cost += (double)w.M * w.N * 2 / kWideStores;
    return cost;
}
bool pair_serves(const PairChoice& c, const TileProduct& x, int x_out, const TileProduct& w, int w_out) {
    if (c.path == PairChoice::SEPARATE || x.N != w.N || x.alpha != w.alpha || x.b_e5m2 || w.b_e5m2 || (!x.mask && !w.mask)) return false;
    if (c.path == PairChoice::PERSISTENT) return persistent_pair_serves(x, x_out, w, w_out);
    return x.K > w.K ? gemm_tile_pair_serves(x, c.kind_x, w, c.kind_w) : gemm_tile_pair_serves(w, c.kind_w, x, c.kind_x);
}
PairChoice choose_pair(const TileProduct& x, const ProductChoice& cx, int x_out, const TileProduct& w, const ProductChoice& cw, int w_out) {
    PairChoice best{PairChoice::SEPARATE, 0, 0};
    const int cus = device_cus();
    const double apart = cx.cost + cw.cost;
    const double one = pair_serves({PairChoice::PERSISTENT, 0, 0}, x, x_out, w, w_out) ? persistent_pair_cost(x, x_out, w, w_out, cus) : 1e30;
    double cost = 1e30;
    if (one < pair_margin(cx, cw) * apart) {
        cost = 1.1 * one;   // it is the more hopeful one of the two estimates
        best = {PairChoice::PERSISTENT, 0, 0};
    }
    for (const PairTile& kx : kPairTiles)
        for (const PairTile& kw : kPairTiles)
            if (pair_serves({PairChoice::TILE, kx.kind, kw.kind}, x, x_out, w, w_out)) {
                const double c = tile_pair_cost(x, x_out, kx, w, w_out, kw, cus);
                if (c < kTilePairMargin * apart && c < cost) {
                    cost = c;
                    best = {PairChoice::TILE, kx.kind, kw.kind};
                }
            }
    return best;
}
hipError_t run_pair(const PairChoice& c, const TileProduct& x, int x_out, const TileProduct& w, int w_out, hipStream_t stream) {
    const bool x_long = x.K > w.K;
    if (c.path == PairChoice::TILE)
        return x_long ? gemm_tile_pair(x, c.kind_x, x_out != BF16, w, c.kind_w, w_out != BF16, stream)
                      : gemm_tile_pair(w, c.kind_w, w_out != BF16, x, c.kind_x, x_out != BF16, stream);
    if (c.path != PairChoice::PERSISTENT) return hipErrorInvalidValue;
    const TileProduct &lng = x_long ? x : w, &sht = x_long ? w : x;
    const int cus = device_cus();
    const auto kind = [](const TileProduct& p, int out) { return !p.mask ? BIG4_PLAIN : out == BF16 ? BIG4_ROTATED : BIG4_WIDE; };
    // a plain product's mask requests, which nothing reads, go to its A
    const auto rot = [](const TileProduct& p) { return RotEpilogue{p.mask ? p.mask : p.a_codes, p.signs.w[0], p.rot_c}; };
    Big4Other o{sht.a_codes, sht.a_scales, sht.b_codes, sht.b_scales, sht.c, rot(sht), sht.M, sht.K, 0,
                kind(sht, x_long ? w_out : x_out), kind(lng, x_long ? x_out : w_out)};
    pair_makespan(lng, sht, cus, &o.rounds);
    const int late = big4_late_start(sht.K, 1), grid = pair_grid(big_tiles(x) + big_tiles(w), cus);
    const auto go_rotated = [&](auto pair, auto hd) {
        constexpr int P = decltype(pair)::value, R = decltype(hd)::value;
        return x.M % 64 || w.M % 64 ? launch_pair_as<P, R, true>(lng, o, rot(lng), late, grid, stream) : launch_pair_as<P, R, false>(lng, o, rot(lng), late, grid, stream);
    };
    const int hd = x.mask ? x.hd : w.hd;
    const auto go = [&](auto pair) {
        if constexpr ((decltype(pair)::value & BIG4_PLAIN) == 0) {   // a plain one comes with blocks of 32
            if (hd == 64) return go_rotated(pair, std::integral_constant<int, 64>{});
            if (hd == 128) return go_rotated(pair, std::integral_constant<int, 128>{});
        }
        return go_rotated(pair, std::integral_constant<int, 32>{});
    };
    switch (o.kind | o.long_kind) {
        case BIG4_ROTATED: return go(std::integral_constant<int, BIG4_ROTATED>{});
        case BIG4_ROTATED | BIG4_WIDE: return go(std::integral_constant<int, BIG4_ROTATED | BIG4_WIDE>{});
        case BIG4_PLAIN | BIG4_ROTATED: return go(std::integral_constant<int, BIG4_PLAIN | BIG4_ROTATED>{});
        case BIG4_PLAIN | BIG4_WIDE: return go(std::integral_constant<int, BIG4_PLAIN | BIG4_WIDE>{});
        default: return hipErrorInvalidValue;
    }
}

// Whether a product on 128 x 128 tiles whose epilogue goes on with what is made of it (`end` us a tile and CU) is expected to beat the
// fastest kernel of the product alone and a pass of its own over its result (us)
bool product_after_pays(const TileProduct& p, double end, double pass) {
    const int cus = device_cus();
    const KernelCost& k = tile_costs(false, TILE_128x128, p.K, 1);
    const double tiles = (double)((p.M + 127) / 128) * ((p.N + 127) / 128);
    return tile_cost(k, p.M, p.N, p.K, 1, cus) + end * tiles / cus < choose_product(p, BF16, BF16, nullptr, 0).cost + pass;
}

TileProduct make_product(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes, const uint8_t* b_scales, int64_t M, int64_t N,
                         int64_t K, float alpha, void* c, int a_layout, int b_layout) {
    TileProduct p{};
    p.a_codes = a_codes; p.a_scales = a_scales; p.b_codes = b_codes; p.b_scales = b_scales; p.c = c;
    p.M = (int)M; p.N = (int)N; p.K = (int)K; p.alpha = alpha; p.hd = 32; p.splits = 1;
    p.a_tiled = a_layout == LAYOUT_TILED; p.b_tiled = b_layout == LAYOUT_TILED;
    return p;
}

hipError_t gemm_mxfp4_tn(const uint8_t* a_codes, const uint8_t* a_scales, const uint8_t* b_codes,
                         const uint8_t* b_scales, int64_t M, int64_t N, int64_t K, float alpha, void* c, int c_dtype,
                         int a_layout, int b_layout, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (M == 0 || N == 0) return hipSuccess;
    if (M >= (1ll << 31) || N >= (1ll << 31) || K >= (1ll << 31)) return hipErrorInvalidValue;
    const TileProduct p = make_product(a_codes, a_scales, b_codes, b_scales, M, N, K, alpha, c, a_layout, b_layout);
    return run_product(choose_product(p, c_dtype, c_dtype, workspace, workspace_bytes), p, c_dtype, c_dtype, workspace, stream);
}

// The product with the rotation in the persistent kernel's epilogue (bf16, Hadamard block 32)
bool gemm_persistent_rotates(const uint8_t* a_scales, const uint8_t* b_scales, int64_t M, int64_t N, int64_t K) {
    return gemm_supports_tiled(M, N, K) && K > 768 && persistent_serves(M, N, K, a_scales, b_scales, nullptr);
}
hipError_t gemm_persistent_rotated(TileProduct p, hipStream_t stream) {
    return run_product({ProductChoice::PERSISTENT, 0, 1, true}, p, BF16, BF16, nullptr, stream);
}

}  // namespace qm
