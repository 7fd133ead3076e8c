// What stands around the product of an evaluated model's logits (gemm_two.hip): the classes' weight rounded to bf16 in the blocks that the product
// reads, and the rows' losses from what it left beside the logits.  Both are bound by HBM, the second at a few thousand rows by latency: 32000 x 640 18.3 us
// (6.7 TB/s, part of it from the memory-side cache; past the caches 24.6), 4096 rows of 334 parts 8.2 (a pass over their logits 49).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qm_kernels.h"
#include "qm_math.h"

namespace qm {

namespace {

constexpr float kLog2e = 1.44269504088896340736f, kLn2 = 0.69314718055994530942f;
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));

// w [V, K] fp32 -> bf16 in [ceil(V / 16)][K / 32][16][64 bytes]: a lane's eight elements of a row, a wave's 1 KiB block; rows past the end are
// not written (the product drops what it makes of them)
__global__ __launch_bounds__(256) void bf16_blocks_kernel(const float* __restrict__ w, int64_t V, int K, int64_t blocks, uint4* __restrict__ out) {
    const int64_t block = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (block >= blocks) return;
    const int lane = threadIdx.x & 63, per_row = K / 32;
    const int64_t row = block / per_row * 16 + (lane >> 2);
    if (row >= V) return;
    const float* src = w + row * K + block % per_row * 32 + (lane & 3) * 8;
    const f4 lo = *reinterpret_cast<const f4*>(src), hi = *(reinterpret_cast<const f4*>(src) + 1);
    const auto two = [](float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, b2)); };
    out[block * 64 + lane] = make_uint4(two(lo[0], lo[1]), two(lo[2], lo[3]), two(hi[0], hi[1]), two(hi[2], hi[3]));
}

// losses[row] from a row's parts: 32 rows a workgroup, eight lanes to a row, in a fixed order
__global__ __launch_bounds__(256) void logits_loss_rows_kernel(const float2* __restrict__ parts, int segments, int T, const uint16_t* __restrict__ logits, int V,
                                                           const int64_t* __restrict__ targets, int64_t ignore, float* __restrict__ losses) {
    __shared__ float2 lds[256];
    const int r = threadIdx.x & 31, part = threadIdx.x >> 5, row = (int)blockIdx.x * 32 + r;
    const auto relative = [](float m, float top) { return __builtin_amdgcn_exp2f(m == -INFINITY ? -INFINITY : (m - top) * kLog2e); };
    float m = -INFINITY, s = 0.0f;
    const auto join = [&](float om, float os) {
        const float top = fmaxf(m, om);
        s = s * relative(m, top) + os * relative(om, top);
        m = top;
    };
    if (row < T) {
        constexpr int kAhead = 8;
        for (int g = part; g < segments; g += 8 * kAhead) {
            float2 v[kAhead];
#pragma unroll
            for (int k = 0; k < kAhead; ++k) v[k] = g + 8 * k < segments ? parts[(int64_t)(g + 8 * k) * T + row] : make_float2(-INFINITY, 0.0f);
#pragma unroll
            for (int k = 0; k < kAhead; ++k) join(v[k].x, v[k].y);
        }
    }
    lds[threadIdx.x] = make_float2(m, s);
    __syncthreads();
    if (part == 0 && row < T) {
#pragma unroll
        for (int k = 1; k < 8; ++k) join(lds[32 * k + r].x, lds[32 * k + r].y);
        const int64_t target = targets[row];
        const bool known = target >= 0 && target < V;
        const float at = known ? u2f((uint32_t)logits[(int64_t)row * V + target] << 16) : 0.0f;
        losses[row] = target == ignore ? 0.0f : known ? (m - at) + __builtin_amdgcn_logf(s) * kLn2 : __builtin_nanf("");
    }
}

}  // namespace

hipError_t bf16_blocks(const float* w, int64_t V, int64_t K, void* out, hipStream_t stream) {
    const int64_t blocks = (V + 15) / 16 * (K / 32);
    bf16_blocks_kernel<<<dim3((unsigned)((blocks + 3) / 4)), dim3(256), 0, stream>>>(w, V, (int)K, blocks, static_cast<uint4*>(out));
    return hipGetLastError();
}
hipError_t logits_loss_rows(const void* parts, int64_t segments, int64_t T, const void* logits, int64_t V, const int64_t* targets, int64_t ignore, float* losses,
                            hipStream_t stream) {
    logits_loss_rows_kernel<<<dim3((unsigned)((T + 31) / 32)), dim3(256), 0, stream>>>(static_cast<const float2*>(parts), (int)segments, (int)T,
                                                                                       static_cast<const uint16_t*>(logits), (int)V, targets, ignore, losses);
    return hipGetLastError();
}

}  // namespace qm
