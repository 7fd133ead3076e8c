// Mean cross-entropy of logits against target classes, forward only: the loss of an evaluated model.
//
// What bounds it: the logits, read once.  As library calls (log-softmax, a conversion to fp32, a reduction over the picked
// entries) 4096 x 32000 bf16 logits went through memory four times: 119 + 125 + 21 us against a floor of 51 us.  Here a
// workgroup reads its row once and keeps a running maximum and the sum of exponentials relative to it per lane, four 16-byte
// requests ahead; the lanes meet in a fixed order.  One small workgroup then adds the rows' losses, also in a fixed order.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "qm_kernels.h"
#include "qm_math.h"
#include "streaming.h"

namespace qm {

namespace {

constexpr int kLossThreads = 256;
constexpr float kLog2e = 1.44269504088896340736f, kLn2 = 0.69314718055994530942f;

// running (maximum m, sum of 2^((x - m) log2 e)); an empty one is (-inf, 0)
struct LogSum {
    float m = -INFINITY, s = 0.0f;
    // a maximum of -inf as the reference of a difference would make NaN of -inf - -inf: those terms are zero
    __device__ __forceinline__ static float relative(float x, float m) {
        return __builtin_amdgcn_exp2f(m == -INFINITY ? -INFINITY : (x - m) * kLog2e);
    }
    template <int N>
    __device__ __forceinline__ void add(const float (&v)[N]) {
        float top = m;
#pragma unroll
        for (int i = 0; i < N; ++i) top = fmaxf(top, v[i]);
        float t = s * relative(m, top);
#pragma unroll
        for (int i = 0; i < N; ++i) t += v[i] != v[i] ? v[i] : relative(v[i], top);   // a NaN stays one
        m = top;
        s = t;
    }
    __device__ __forceinline__ void join(float om, float os) {
        const float top = fmaxf(m, om);
        s = s * relative(m, top) + os * relative(om, top);
        m = top;
    }
};

template <typename T>
__device__ __forceinline__ void widen(const uint4& raw, float (&v)[16 / sizeof(T)]) {
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
    if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = u2f(w[i] << 16);
            v[2 * i + 1] = u2f(w[i] & 0xffff0000u);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = u2f(w[i]);
    }
}
__device__ __forceinline__ float widen(uint16_t x) { return u2f((uint32_t)x << 16); }
__device__ __forceinline__ float widen(float x) { return x; }

// losses[row] = log(sum exp(logits[row])) - logits[row][target], 0 for an ignored row; a target that is no class: NaN
// STREAM: requests past the caches.  4096 x 32000 bf16 57 -> 48.5 us (5.4 TB/s), 600 x 32000 13.0 -> 13.3
template <typename T, bool STREAM>
__global__ __launch_bounds__(kLossThreads) void cross_entropy_rows_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
                                                                          int64_t classes, int64_t ignore, float* __restrict__ losses) {
    constexpr int kPer = 16 / sizeof(T), kAhead = 4;
    __shared__ float lds_m[kLossThreads / 64], lds_s[kLossThreads / 64];
    const int64_t row = blockIdx.x;
    const int64_t target = targets[row];
    if (target == ignore) {   // uniform
        if (threadIdx.x == 0) losses[row] = 0.0f;
        return;
    }
    const T* x = logits + row * classes;
    // rows start at any element: a head up to the first 16-byte boundary and a tail, one element per lane
    int64_t head = (int64_t)((16 - (reinterpret_cast<uintptr_t>(x) & 15)) & 15) / (int64_t)sizeof(T);
    head = head < classes ? head : classes;
    const int64_t pieces = (classes - head) / kPer, tail = head + pieces * kPer;
    const uint4* p = reinterpret_cast<const uint4*>(x + head);
    LogSum acc;
    int64_t i = threadIdx.x;
    for (; i + (kAhead - 1) * kLossThreads < pieces; i += kAhead * kLossThreads) {
        uint4 raw[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) raw[j] = STREAM ? stream_load(p + i + j * kLossThreads) : p[i + j * kLossThreads];
        float v[kAhead * kPer];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            float part[kPer];
            widen<T>(raw[j], part);
#pragma unroll
            for (int e = 0; e < kPer; ++e) v[j * kPer + e] = part[e];
        }
        acc.add(v);
    }
    for (; i < pieces; i += kLossThreads) {
        float v[kPer];
        widen<T>(p[i], v);
        acc.add(v);
    }
    const int64_t single = (int64_t)threadIdx.x < head ? (int64_t)threadIdx.x : tail + (int64_t)threadIdx.x - head;   // head and tail: fewer than 16 elements
    if (single < classes) {
        const float v[1] = {widen(x[single])};
        acc.add(v);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) acc.join(__shfl_xor(acc.m, d), __shfl_xor(acc.s, d));
    if ((threadIdx.x & 63) == 0) {
        lds_m[threadIdx.x >> 6] = acc.m;
        lds_s[threadIdx.x >> 6] = acc.s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        LogSum all;
#pragma unroll
        for (int w = 0; w < kLossThreads / 64; ++w) all.join(lds_m[w], lds_s[w]);
        const bool known = target >= 0 && target < classes;
        losses[row] = known ? (all.m - widen(x[target])) + __builtin_amdgcn_logf(all.s) * kLn2 : __builtin_nanf("");
    }
}

// mean over the rows that are not ignored: each lane adds every 1024th row, then pairwise.  No such row: 0 / 0, as the library
__global__ __launch_bounds__(1024) void cross_entropy_mean_kernel(const float* __restrict__ losses, const int64_t* __restrict__ targets, int64_t rows,
                                                                  int64_t ignore, float* __restrict__ loss) {
    __shared__ float sums[1024];
    __shared__ float counts[1024];
    float sum = 0.0f;
    int64_t count = 0;
    for (int64_t r = threadIdx.x; r < rows; r += 1024) {
        sum += losses[r];
        count += targets[r] != ignore;
    }
    sums[threadIdx.x] = sum;
    counts[threadIdx.x] = (float)count;
    __syncthreads();
    for (int d = 512; d > 0; d >>= 1) {
        if ((int)threadIdx.x < d) {
            sums[threadIdx.x] += sums[threadIdx.x + d];
            counts[threadIdx.x] += counts[threadIdx.x + d];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = sums[0] / counts[0];
}

}  // namespace

hipError_t loss_mean(const float* losses, const int64_t* targets, int64_t rows, int64_t ignore, float* loss, hipStream_t stream) {
    cross_entropy_mean_kernel<<<dim3(1), dim3(1024), 0, stream>>>(losses, targets, rows, ignore, loss);
    return hipGetLastError();
}

hipError_t cross_entropy_mean(const void* logits, int dtype, const int64_t* targets, int64_t rows, int64_t classes, int64_t ignore,
                              float* losses, float* loss, hipStream_t stream) {
    const auto go = [&](const auto* x, auto past) {
        using T = std::remove_const_t<std::remove_pointer_t<decltype(x)>>;
        constexpr int64_t kRows = 1 << 23;   // of a launch: a grid has fewer than 2^32 threads
        for (int64_t r = 0; r < rows; r += kRows)
            cross_entropy_rows_kernel<T, decltype(past)::value><<<dim3((unsigned)(rows - r < kRows ? rows - r : kRows)), dim3(kLossThreads), 0, stream>>>(
                x + r * classes, targets + r, classes, ignore, losses + r);
    };
    const auto by_size = [&](const auto* x) {
        if (rows * classes * (int64_t)sizeof(*x) >= kPastTheCaches) go(x, std::true_type{});
        else go(x, std::false_type{});
    };
    if (rows > 0) {
        if (dtype == BF16) by_size(static_cast<const uint16_t*>(logits));
        else by_size(static_cast<const float*>(logits));
    }
    return loss_mean(losses, targets, rows, ignore, loss, stream);
}

}  // namespace qm
