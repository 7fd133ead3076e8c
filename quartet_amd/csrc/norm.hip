// RMSNorm of an evaluated model's last hidden state (src/models/llama.py:64-75 of the reference), with the residual sum in front of it: what
// feeds the unquantized lm_head.  out = (x + add) / sqrt(mean((x + add)^2) + eps) * gain, in fp32, stored in the dtype that the next
// layer reads.
//
// One wave per row, which it keeps in registers: a lane takes four consecutive elements every 256.  The mean is an fp32 sum of the
// lanes' sums.  What bounds it: HBM, and latency at a few thousand rows.  4096 x 640 with a bf16 summand and bf16 out: seven
// library kernels took 43 us, this one 6.8.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "qm_kernels.h"
#include "qm_math.h"

namespace qm {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef uint32_t w2 __attribute__((ext_vector_type(2)));

// blocks: the result goes to blocks of 16 rows and 32 elements, [rows / 16][cols / 32][16][32], as the product of the logits reads it (gemm_two.hip).
// NV: vectors of four per lane, cols <= 256 NV; cols % 4 == 0.  TA: void, uint16_t (bf16) or float
template <int NV, typename TA, typename TOut>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const float* __restrict__ x, const TA* __restrict__ add, const float* __restrict__ gain, float eps,
                                                           int64_t rows, int cols, TOut* __restrict__ out, int blocks) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;   // a whole wave
    f4 v[NV];
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = i * 256 + lane * 4;
        v[i] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        if (c < cols) {
            v[i] = *reinterpret_cast<const f4*>(x + row * cols + c);
            if constexpr (std::is_same<TA, float>::value) {
                v[i] = v[i] + *reinterpret_cast<const f4*>(add + row * cols + c);
            } else if constexpr (std::is_same<TA, uint16_t>::value) {
                const w2 a = *reinterpret_cast<const w2*>(add + row * cols + c);
                v[i] = v[i] + f4{u2f(a[0] << 16), u2f(a[0] & 0xffff0000u), u2f(a[1] << 16), u2f(a[1] & 0xffff0000u)};
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) sum = sum + ((v[i][0] * v[i][0] + v[i][1] * v[i][1]) + (v[i][2] * v[i][2] + v[i][3] * v[i][3]));
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) sum = sum + __shfl_xor(sum, m, 64);
    const float f = 1.0f / __builtin_sqrtf(sum / (float)cols + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = i * 256 + lane * 4;
        if (c >= cols) continue;
        const f4 r = v[i] * f * *reinterpret_cast<const f4*>(gain + c);
        const int64_t at = blocks ? (row >> 4) * 16 * cols + (c >> 5) * 512 + (row & 15) * 32 + (c & 31) : row * cols + c;
        if constexpr (sizeof(TOut) == 2)
            *reinterpret_cast<w2*>(out + at) =
                w2{__builtin_bit_cast(uint32_t, __builtin_convertvector(f2{r[0], r[1]}, b2)), __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{r[2], r[3]}, b2))};
        else
            *reinterpret_cast<f4*>(out + at) = r;
    }
}

}  // namespace

// cols % 4 == 0, cols <= 4096; x, gain, out (fp32) and an fp32 summand 16-byte, bf16 ones 8-byte aligned
hipError_t rmsnorm_rows(const float* x, const void* add, int add_dtype, const float* gain, float eps, int64_t rows, int64_t cols, void* out, int out_dtype,
                        hipStream_t stream, bool blocks) {
    constexpr int64_t kRows = 1 << 25;   // of a launch: a grid has fewer than 2^32 threads, 64 a row
    const auto go = [&](auto nv, const auto* a, auto* o) {
        for (int64_t r = 0; r < rows; r += kRows) {
            using A = std::remove_const_t<std::remove_pointer_t<decltype(a)>>;
            const A* ar = nullptr;
            if constexpr (!std::is_void<A>::value) ar = a + r * cols;
            const int64_t n = rows - r < kRows ? rows - r : kRows;
            rmsnorm_rows_kernel<decltype(nv)::value><<<dim3((unsigned)((n + 3) / 4)), dim3(256), 0, stream>>>(x + r * cols, ar, gain, eps, n, (int)cols, o + r * cols, (int)blocks);
        }
    };
    const auto by_out = [&](auto nv, const auto* a) {
        if (out_dtype == BF16) go(nv, a, static_cast<uint16_t*>(out));
        else go(nv, a, static_cast<float*>(out));
    };
    const auto by_add = [&](auto nv) {
        if (!add) by_out(nv, static_cast<const void*>(nullptr));
        else if (add_dtype == BF16) by_out(nv, static_cast<const uint16_t*>(add));
        else by_out(nv, static_cast<const float*>(add));
    };
    if (cols <= 768) by_add(std::integral_constant<int, 3>{});
    else if (cols <= 1536) by_add(std::integral_constant<int, 6>{});
    else by_add(std::integral_constant<int, 16>{});
    return hipGetLastError();
}

}  // namespace qm
