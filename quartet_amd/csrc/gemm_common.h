// Pieces shared by the FP4 x FP4 product kernels (gemm.hip, gemm_tile.hip): operand geometry, direct global -> LDS
// requests, accumulator read-out and the XCD-aware tile order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "lds_requests.h"
#include "qm_kernels.h"
#include "qm_math.h"

namespace qm {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

constexpr int kBK = 128;             // K elements per step
constexpr int kRowBytes = kBK / 2;   // 64 bytes of codes per row per step

// acc element e of a 32x32 tile is row 8*(e/4) + 4*half + e%4, column lane%32: per store instruction the
// two half-waves each write one 64-byte (bf16) row segment.  rows_left: rows of the block that lie inside the matrix.  (Making a lane's 4 values contiguous along n by
// swapping the MFMA operand roles was measured slower: 64 scattered 8-byte pieces per instruction.)
// One accumulator register into a vector register, in program order: left to itself the compiler copies ten blocks of
// sixteen ahead of the first pass, and the 160 registers that takes push values the K loop needs out to scratch memory,
// whose reloads then wait for every operand load in flight (loads return in order).
__device__ __forceinline__ float acc_read(float a) {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
    return v;
}
// The hazard recogniser does not look inside assembly statements: a matrix instruction's result may be read by a vector
// instruction only a number of wait states after it issued (19 for the sixteen-pass forms).  Every epilogue that reads
// accumulators through acc_read() starts with this, whatever the scheduler has put between the last product and it.
__device__ __forceinline__ void acc_settle() { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory"); }
template <typename OutT, bool IN_ORDER = false>
__device__ __forceinline__ void store_tile(const v16f& t, float alpha, OutT* __restrict__ c, int64_t row0, int64_t col,
                                           int64_t N, int half, int rows_left = 32) {
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        const int rl = 8 * (e / 4) + 4 * half + (e & 3);
        const int64_t r = row0 + rl;
        const float v0 = (IN_ORDER ? acc_read(t[e]) : t[e]) * alpha, v1 = (IN_ORDER ? acc_read(t[e + 1]) : t[e + 1]) * alpha;
        if constexpr (sizeof(OutT) == 2) {
            // v_cvt_pk_bf16_f32: round-to-nearest-even, two values per instruction
            const v2bf p = __builtin_convertvector(v2f{v0, v1}, v2bf);
            const uint32_t bits = __builtin_bit_cast(uint32_t, p);
            if (rl < rows_left) c[r * N + col] = (uint16_t)(bits & 0xffffu);
            if (rl + 1 < rows_left) c[(r + 1) * N + col] = (uint16_t)(bits >> 16);
        } else {
            if (rl < rows_left) c[r * N + col] = v0;
            if (rl + 1 < rows_left) c[(r + 1) * N + col] = v1;
        }
    }
}

// Item order: workgroup ids are dealt round-robin to the 8 XCDs by the hardware; give each XCD a contiguous run of items, of any
// number of them, K ranges of a product being runs of tiles one after the other.
__device__ __forceinline__ int xcd_run(int id, int total) {
    const int xcd = id & 7, rest = total & 7;
    return xcd * (total >> 3) + (xcd < rest ? xcd : rest) + (id >> 3);
}
// Tile order: groups of GM tile rows (about a thousand matrix rows), column by column, so that the tiles of a run, which share an
// L2, also share A and B panels.
template <int GM = 4>
__device__ __forceinline__ void tile_of_run(int t, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int per_group = GM * tiles_n;
    const int group = t / per_group;
    const int first_m = group * GM;
    const int gm = (tiles_m - first_m) < GM ? (tiles_m - first_m) : GM;
    const int r = t - group * per_group;
    tm = first_m + r % gm;
    tn = r / gm;
}

// one MFMA, then one memory instruction of the given class, n times: keeps the matrix pipe fed while the
// wave issues its LDS / VMEM instructions
#define QM_SCHED_PAIR(mask, n)                                   \
    for (int _i = 0; _i < (n); ++_i) {                           \
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       \
        __builtin_amdgcn_sched_group_barrier((mask), 1, 0);      \
    }

// hipFuncSetAttribute(MaxDynamicSharedMemorySize) once per kernel and device instead of on every launch
constexpr int kMaxDevices = 64;
template <typename Kern>
hipError_t allow_dynamic_lds(Kern kern, int bytes, std::atomic<bool> (&done)[kMaxDevices]) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < kMaxDevices && done[dev].load(std::memory_order_acquire)) return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && dev >= 0 && dev < kMaxDevices) done[dev].store(true, std::memory_order_release);
    return e;
}

int device_cus() {
    static int cached = 0;  // one GPU model per process
    if (cached > 0) return cached;
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        n > 0)
        return cached = n;
    return 256;
}

}  // namespace
}  // namespace qm
