// Causal attention of bf16 heads, forward only: what an evaluated model runs between its attention projections.
//
// What bounds it: at 8 x 512 tokens and 5 heads of 128 latency (1.3 GFLOP of unmasked products, 21 MB), at long sequences the
// matrix pipe and the exponentials.  The library's kernel took 34 us there plus a fill of 4.4 us.
//
// A workgroup of four waves owns 64 * QB queries of one head, a wave 16 * QB of them; the keys and values of 64 positions at
// a time go through LDS, the next 64 on their way into registers meanwhile.  Both products have the queries as the
// columns of v_mfma_f32_16x16x32_bf16: S^T = K Q^T leaves a lane with scores of one query (lane % 16) against keys
// 4 (lane / 16) + e of each block of sixteen, and that is, up to an order of the contraction which V^T follows, the operand
// layout of O^T = V^T P^T: probabilities never cross lanes.  V is transposed four keys at a time on its way into LDS.
// Scores, the running maximum, the probabilities' sum and the output accumulate in fp32; probabilities enter the second
// product as bf16, as in the library's kernel.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qm_kernels.h"
#include "qm_math.h"

namespace qm {

namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kKeys = 64;   // positions per step

__device__ __forceinline__ v8bf as_v8bf(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(v8bf, make_uint4(a, b, c, d));
}
// over the four lanes that share lane % 16
template <typename F>
__device__ __forceinline__ float across_quarters(float v, F&& f) {
    const auto a = __builtin_amdgcn_permlane16_swap(f2u(v), f2u(v), false, false);
    v = f(u2f(a[0]), u2f(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(f2u(v), f2u(v), false, false);
    return f(u2f(b[0]), u2f(b[1]));
}

// q, k, v, out: [batch, S, heads, D] contiguous
template <int D, int QB>
__global__ __launch_bounds__(256) void attention_causal_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                                               const uint16_t* __restrict__ v, uint16_t* __restrict__ out, int S, int heads,
                                                               int all_heads, int heads_per_xcd, int q_blocks, float scale_log2e) {
    constexpr int kRows = 64 * QB;                       // queries of the workgroup
    constexpr int kKPitch = D * 2 + 16;                  // bytes per key row in LDS: rows four banks apart
    constexpr int kVPitch = kKeys * 2 + 16;              // bytes per row (one d) of the transposed values
    constexpr int kPieces = D / 8;                       // 16-byte pieces per row
    constexpr int kKLoads = kKeys * kPieces / 256;       // per lane and step
    constexpr int kVUnits = kKeys / 4 * kPieces;         // four keys x eight d each
    static_assert(kKeys * kPieces % 256 == 0 && kVUnits <= 256, "one unit of V per lane");
    __shared__ __align__(16) uint8_t lds[kKeys * kKPitch + D * kVPitch];
    uint8_t* const lds_k = lds;
    uint8_t* const lds_v = lds + kKeys * kKPitch;

    // workgroups of one head share an XCD and its L2; the longest rows of queries start first
    const int x = (int)blockIdx.x & 7, rest = (int)blockIdx.x >> 3;
    const int head = x + 8 * (rest % heads_per_xcd), q0 = (q_blocks - 1 - rest / heads_per_xcd) * kRows;
    if (head >= all_heads) return;   // the whole workgroup
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, g = lane >> 4;
    const int64_t pitch = (int64_t)heads * D;            // elements from one position to the next
    const int64_t base = (int64_t)(head / heads) * S * pitch + (int64_t)(head % heads) * D;
    const int w0 = q0 + wave * 16 * QB;                  // the wave's first query

    uint4 qf[QB][D / 32];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
        const int row = w0 + b * 16 + col < S ? w0 + b * 16 + col : S - 1;   // a query past the end repeats the last one and is not stored
#pragma unroll
        for (int c = 0; c < D / 32; ++c) qf[b][c] = *reinterpret_cast<const uint4*>(q + base + row * pitch + c * 32 + g * 8);
    }
    uint4 kr[kKLoads], vr[4];
    const int kg = tid & 15, oct = tid >> 4;             // this lane's unit of V
    const auto request = [&](int k0) {
#pragma unroll
        for (int j = 0; j < kKLoads; ++j) {
            const int piece = tid + 256 * j, key = k0 + piece / kPieces;
            kr[j] = *reinterpret_cast<const uint4*>(k + base + (key < S ? key : S - 1) * pitch + piece % kPieces * 8);
        }
        if (kVUnits == 256 || tid < kVUnits) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = k0 + kg * 4 + i;
                vr[i] = *reinterpret_cast<const uint4*>(v + base + (key < S ? key : S - 1) * pitch + oct * 8);
            }
        }
    };
    const auto stage = [&] {
#pragma unroll
        for (int j = 0; j < kKLoads; ++j) {
            const int piece = tid + 256 * j;
            *reinterpret_cast<uint4*>(lds_k + piece / kPieces * kKPitch + piece % kPieces * 16) = kr[j];
        }
        if (kVUnits == 256 || tid < kVUnits) {
            const uint32_t r[4][4] = {{vr[0].x, vr[0].y, vr[0].z, vr[0].w}, {vr[1].x, vr[1].y, vr[1].z, vr[1].w},
                                      {vr[2].x, vr[2].y, vr[2].z, vr[2].w}, {vr[3].x, vr[3].y, vr[3].z, vr[3].w}};
#pragma unroll
            for (int i = 0; i < 4; ++i) {   // d = 8 oct + 2 i and the one after it
                uint8_t* dst = lds_v + (oct * 8 + 2 * i) * kVPitch + kg * 8;
                *reinterpret_cast<uint2*>(dst) = make_uint2((r[0][i] & 0xffffu) | (r[1][i] << 16), (r[2][i] & 0xffffu) | (r[3][i] << 16));
                *reinterpret_cast<uint2*>(dst + kVPitch) = make_uint2((r[0][i] >> 16) | (r[1][i] & 0xffff0000u), (r[2][i] >> 16) | (r[3][i] & 0xffff0000u));
            }
        }
    };

    v4f o[QB][D / 16];
    float top[QB], sum[QB];   // running maximum of the scaled scores (log2), this lane's share of the sum
#pragma unroll
    for (int b = 0; b < QB; ++b) {
        top[b] = -INFINITY;
        sum[b] = 0.0f;
#pragma unroll
        for (int d = 0; d < D / 16; ++d) o[b][d] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const int keys = q0 + kRows < S ? q0 + kRows : S;
    request(0);
    for (int k0 = 0; k0 < keys; k0 += kKeys) {
        __syncthreads();   // every wave has read the step before
        stage();
        __syncthreads();
        if (k0 + kKeys < keys) request(k0 + kKeys);
        if (k0 > w0 + 16 * QB - 1) continue;   // all keys lie behind the wave's queries
        v4f s[QB][kKeys / 16];
#pragma unroll
        for (int t = 0; t < kKeys / 16; ++t) {
#pragma unroll
            for (int b = 0; b < QB; ++b) s[b][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int c = 0; c < D / 32; ++c) {
                const v8bf kf = __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4*>(lds_k + (t * 16 + col) * kKPitch + c * 64 + g * 16));
#pragma unroll
                for (int b = 0; b < QB; ++b)
                    s[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, __builtin_bit_cast(v8bf, qf[b][c]), s[b][t], 0, 0, 0);
            }
        }
        v8bf p[QB][kKeys / 32];
#pragma unroll
        for (int b = 0; b < QB; ++b) {
            const int query = w0 + b * 16 + col;
            float m = top[b];
#pragma unroll
            for (int t = 0; t < kKeys / 16; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float z = s[b][t][e] * scale_log2e;
                    // a key past the end (read as the last one) lies behind every query that is stored
                    s[b][t][e] = k0 + t * 16 + 4 * g + e <= query ? z : -INFINITY;
                    m = fmaxf(m, s[b][t][e]);
                }
            m = across_quarters(m, [](float a, float c) { return fmaxf(a, c); });
            const float shrink = __builtin_amdgcn_exp2f(top[b] - m);   // 0 on the first step
            top[b] = m;
            float part = 0.0f;
            uint32_t w[kKeys / 16][2];
#pragma unroll
            for (int t = 0; t < kKeys / 16; ++t) {
                float e4[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    e4[e] = __builtin_amdgcn_exp2f(s[b][t][e] - m);
                    part += e4[e];
                }
                w[t][0] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{e4[0], e4[1]}, v2bf));
                w[t][1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{e4[2], e4[3]}, v2bf));
            }
            sum[b] = sum[b] * shrink + part;
#pragma unroll
            for (int u = 0; u < kKeys / 32; ++u) p[b][u] = as_v8bf(w[2 * u][0], w[2 * u][1], w[2 * u + 1][0], w[2 * u + 1][1]);
#pragma unroll
            for (int d = 0; d < D / 16; ++d) o[b][d] *= shrink;
        }
        // contraction slots of a lane: keys 32 u + 4 g .. + 3, then 32 u + 16 + 4 g .. + 3
#pragma unroll
        for (int d = 0; d < D / 16; ++d)
#pragma unroll
            for (int u = 0; u < kKeys / 32; ++u) {
                const uint8_t* src = lds_v + (d * 16 + col) * kVPitch + u * 64 + g * 8;
                const uint2 lo = *reinterpret_cast<const uint2*>(src), hi = *reinterpret_cast<const uint2*>(src + 32);
                const v8bf vf = as_v8bf(lo.x, lo.y, hi.x, hi.y);
#pragma unroll
                for (int b = 0; b < QB; ++b) o[b][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p[b][u], o[b][d], 0, 0, 0);
            }
    }
#pragma unroll
    for (int b = 0; b < QB; ++b) {
        const int query = w0 + b * 16 + col;
        const float inv = 1.0f / across_quarters(sum[b], [](float a, float c) { return a + c; });
        if (query < S) {
            uint16_t* dst = out + base + query * pitch + 4 * g;
#pragma unroll
            for (int d = 0; d < D / 16; ++d) {
                const v4f r = o[b][d] * inv;
                const v2bf r0 = __builtin_convertvector(v2f{r[0], r[1]}, v2bf), r1 = __builtin_convertvector(v2f{r[2], r[3]}, v2bf);
                *reinterpret_cast<uint2*>(dst + d * 16) = make_uint2(__builtin_bit_cast(uint32_t, r0), __builtin_bit_cast(uint32_t, r1));
            }
        }
    }
}

template <int D, int QB>
void launch_attention(const void* q, const void* k, const void* v, void* out, int64_t batch, int64_t S, int64_t heads, hipStream_t stream) {
    const int all = (int)(batch * heads), per_xcd = (all + 7) / 8, q_blocks = (int)((S + 64 * QB - 1) / (64 * QB));
    attention_causal_kernel<D, QB><<<dim3((unsigned)(8 * per_xcd * q_blocks)), dim3(256), 0, stream>>>(
        static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v), static_cast<uint16_t*>(out), (int)S,
        (int)heads, all, per_xcd, q_blocks, (float)(1.4426950408889634 / __builtin_sqrt((double)D)));
}

}  // namespace

bool attention_causal_serves(int64_t batch, int64_t S, int64_t heads, int head_dim) {
    return (head_dim == 64 || head_dim == 128) && batch > 0 && S > 0 && heads > 0 && S < (1 << 24) && batch * heads < (1 << 24) &&
           (batch * heads + 7) / 8 * 8 * ((S + 63) / 64) < (1ll << 31);
}
hipError_t attention_causal(const void* q, const void* k, const void* v, void* out, int64_t batch, int64_t S, int64_t heads, int head_dim,
                            hipStream_t stream) {
    if (!attention_causal_serves(batch, S, heads, head_dim)) return hipErrorInvalidValue;
    const bool wide = batch * heads * ((S + 127) / 128) >= 512;
    if (head_dim == 128) {
        if (wide) launch_attention<128, 2>(q, k, v, out, batch, S, heads, stream);
        else launch_attention<128, 1>(q, k, v, out, batch, S, heads, stream);
    } else {
        if (wide) launch_attention<64, 2>(q, k, v, out, batch, S, heads, stream);
        else launch_attention<64, 1>(q, k, v, out, batch, S, heads, stream);
    }
    return hipGetLastError();
}

}  // namespace qm
