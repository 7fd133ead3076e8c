// The masked inverse rotation of the straight-through backward on eight consecutive elements per lane, shared by the
// stand-alone kernel (hadamard_bwd.hip) and the product kernels that carry it in their epilogue (gemm_tile.hip): the same
// operations in the same order, so the two give the same bits.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qm_kernels.h"
#include "qm_math.h"

namespace qm {
namespace {

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return u2f((uint32_t)__builtin_amdgcn_mov_dpp((int)f2u(v), CTRL, 0xF, 0xF, true));
}
// the value of lane ^ LANE_MASK, without a trip through LDS (by __shfl_xor the product 8192 x 1536 x 4608 with blocks of 128 in
// its epilogue took 52.8 us, now 48.3)
template <int LANE_MASK>
__device__ __forceinline__ float lane_xor(float v) {
    if constexpr (LANE_MASK == 1) return dpp<0xB1>(v);
    else if constexpr (LANE_MASK == 2) return dpp<0x4E>(v);
    else if constexpr (LANE_MASK == 4) return dpp<0x1B>(dpp<0x141>(v));   // the half row mirrored (^ 7), then every quad (^ 3)
    else return dpp<0x128>(v);                                            // 8: the row of sixteen rotated by eight
}
template <int LANE_MASK>
__device__ __forceinline__ void octet_cross_lane_stage(float (&v)[8], int lane_in_chunk) {
    // lower lane of a butterfly: own + partner; upper lane: partner - own = partner + (-own)
    const uint32_t flip = (lane_in_chunk & LANE_MASK) ? 0x80000000u : 0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float p = lane_xor<LANE_MASK>(v[i]);
        v[i] = p + u2f(f2u(v[i]) ^ flip);
    }
}

// v: eight consecutive elements, keep: their mask bits, lic: the lane's octet within its Hadamard block (lane % (HD / 8)).
// Leaves ((v * mask) sign) H / c, the butterfly sums before the multiplication by c.
template <int HD>
__device__ __forceinline__ void octet_inverse_rotation(float (&v)[8], uint32_t keep, int lic, const SignBits& sb) {
    // the block's sign word of this octet by selects: an indexed kernel argument would live in scratch memory
    const uint32_t w0 = sb.w[0], w1 = sb.w[1], w2 = sb.w[2], w3 = sb.w[3];
    uint32_t word = w0;
    if constexpr (HD >= 64) word = (lic & 4) ? w1 : w0;
    if constexpr (HD >= 128) word = (lic & 8) ? ((lic & 4) ? w3 : w2) : word;
    const uint32_t sign8 = (word >> (8 * (lic & 3))) & 0xffu;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        // g * mask as the reference multiplies: the factor is the float 1.0 or 0.0 built from the bit
        const uint32_t all = (uint32_t)__builtin_amdgcn_sbfe((int)keep, i, 1);  // 0 or ~0
        const float x = v[i] * u2f(all & 0x3f800000u);
        v[i] = u2f(f2u(x) ^ (((sign8 >> i) & 1u) << 31));
    }
#pragma unroll
    for (int h = 1; h < 8; h <<= 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (i & h) continue;
            const float a = v[i], b = v[i + h];
            v[i] = a + b;
            v[i + h] = a - b;
        }
    }
    octet_cross_lane_stage<1>(v, lic);
    octet_cross_lane_stage<2>(v, lic);
    if constexpr (HD >= 64) octet_cross_lane_stage<4>(v, lic);
    if constexpr (HD >= 128) octet_cross_lane_stage<8>(v, lic);
}

}  // namespace
}  // namespace qm
