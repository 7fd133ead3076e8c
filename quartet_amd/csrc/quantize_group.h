// The MX group quantizer of one lane: 32 values in registers -> rotation, statistics, scale, FP4 codes, clip mask.  Its
// arithmetic and what bounds it are described at the top of quantize_group.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qm_kernels.h"
#include "qm_math.h"

namespace qm {

namespace {

typedef float v2f __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void butterfly32(float (&v)[32]) {
#pragma unroll
    for (int h = 1; h < 32; h <<= 1) {
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            if (i & h) continue;
            const float a = v[i], b = v[i + h];
            v[i] = a + b;
            v[i + h] = a - b;
        }
    }
}

// pairwise tree: adjacent pairs, then pairs of pairs, ... (the canonical order of the group sums)
__device__ __forceinline__ float tree_sum32(const float (&p)[32]) {
    float t[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) t[i] = p[2 * i] + p[2 * i + 1];
#pragma unroll
    for (int n = 8; n >= 1; n >>= 1)
#pragma unroll
        for (int i = 0; i < n; ++i) t[i] = t[2 * i] + t[2 * i + 1];
    return t[0];
}

struct GroupCodes {
    uint32_t w[4];        // 32 nibbles, element i in bits [4(i%8), +4) of word i/8
    uint32_t scale_byte;  // E8M0
    uint32_t keep;        // bit i = |t_i| < 6
    float deq_scale;      // what a code value is multiplied by in the de-quantized tensor
};

// v_cvt_scalef32_sr_pk_fp4_f32 replaces byte SEL of its destination and keeps the other three, but the
// compiler builtin of this toolchain does not tie the destination to its `old` operand (the untouched bytes
// come back as whatever the allocated register held), so the instruction is issued directly.
template <int SEL>
__device__ __forceinline__ void sr_convert_pair(uint32_t& dst, v2f pair, uint32_t rnd, float scale) {
    if constexpr (SEL == 0) asm("v_cvt_scalef32_sr_pk_fp4_f32 %0, %1, %2, %3" : "+v"(dst) : "v"(pair), "v"(rnd), "v"(scale));
    else if constexpr (SEL == 1) asm("v_cvt_scalef32_sr_pk_fp4_f32 %0, %1, %2, %3 op_sel:[0,0,1,0]" : "+v"(dst) : "v"(pair), "v"(rnd), "v"(scale));
    else if constexpr (SEL == 2) asm("v_cvt_scalef32_sr_pk_fp4_f32 %0, %1, %2, %3 op_sel:[0,0,0,1]" : "+v"(dst) : "v"(pair), "v"(rnd), "v"(scale));
    else asm("v_cvt_scalef32_sr_pk_fp4_f32 %0, %1, %2, %3 op_sel:[0,0,1,1]" : "+v"(dst) : "v"(pair), "v"(rnd), "v"(scale));
}

// the integer form of below_ties() (the bit pattern b becomes (b - 1) | 1): for groups with infinite statistics, where the
// fused form would make an infinity a NaN
__device__ __forceinline__ float below_ties_any(float v) {
    const float w = v + 0.0f;   // both zeros become +0
    return u2f(__builtin_elementwise_sub_sat(f2u(w), 1u) | 1u);
}

// n: the NEGATED rotated group.  The sign rule "negative unless g > 0" makes both zeros negative; on the negated values it reads
// "positive unless n < 0", and the arithmetic in front of the converts turns zeros of either sign into +0 by itself (x y + z
// with two exact zeros of opposite sign), so it costs one XOR of the sign bits of eight codes.  Everything else is symmetric but for
// NaNs, which keep their sign where numbers are negated: their codes are the largest magnitude (the converts') of either sign.

// clip mask, most significant element first so that element 0 lands in bit 0: the sign of |t| - 6 scale (never set for a NaN;
// |t| = 6 scale gives +0), shifted in by a funnel shift.  The subtraction issues at twice the rate of a compare and nothing
// passes through the carry flag: 218 cycles a group against 286 for compare and add-with-carry.  Two chains of sixteen: the
// shifts of one depend on each other.
template <class F>
__device__ __forceinline__ uint32_t clip_mask(const float (&n)[32], float thr, F&& t_of) {
    uint32_t lo = 0u, hi = 0u;
#pragma unroll
    for (int i = 15; i >= 0; --i) {
        lo = __builtin_amdgcn_alignbit(lo, f2u(fabsf(t_of(n[i])) - thr), 31);
        hi = __builtin_amdgcn_alignbit(hi, f2u(fabsf(t_of(n[i + 16])) - thr), 31);
    }
    return (hi << 16) | lo;
}
// The 32 codes; t_of(n) is the value a convert sees, formed next to it: as an array of its own it would hold 32 more registers.
template <class F>
__device__ __forceinline__ void rtn_codes(const float (&n)[32], float hw_scale, F&& t_of, uint32_t (&codes)[4]) {
    // the converts' byte selector must be a literal, hence the macros
#define QM_RTN_PAIR(B) w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, t_of(n[wi * 8 + 2 * (B)]), t_of(n[wi * 8 + 2 * (B) + 1]), hw_scale, (B));
#pragma unroll
    for (int wi = 0; wi < 4; ++wi) {
        uint32_t w = 0u;
        QM_RTN_PAIR(0) QM_RTN_PAIR(1) QM_RTN_PAIR(2) QM_RTN_PAIR(3)
        codes[wi] = w ^ 0x88888888u;
    }
#undef QM_RTN_PAIR
}
template <class F>
__device__ __forceinline__ void sr_codes(const float (&n)[32], float hw_scale, uint64_t seed, int64_t group_index, F&& t_of, uint32_t (&codes)[4]) {
    // element j of a Philox call (16 elements): its random field is the top 22 bits of word j/4 rotated left by
    // 8 * (j%4).  The convert reads the field of a pair's first element from bits 31..10 of its random operand and that of
    // the second from bits 30..9, so the even element's operand is the word rotated by 0 or 16 bits and the odd element's
    // the word rotated by 7 or 23 (one more bit to the right): one v_alignbit_b32 each, none for a word's first element.
#define QM_SR_PAIR(B, J0)                                                                                 \
    {                                                                                                     \
        const uint32_t pw = ph.w[(J0) >> 2];                                                              \
        const uint32_t r_even = ((J0) & 3) == 0 ? pw : __builtin_amdgcn_alignbit(pw, pw, 16);             \
        const uint32_t r_odd = __builtin_amdgcn_alignbit(pw, pw, ((J0) & 3) == 0 ? 25 : 9);               \
        const v2f pr = {t_of(n[wi * 8 + 2 * (B)]), t_of(n[wi * 8 + 2 * (B) + 1])};                        \
        sr_convert_pair<(B)>(even, pr, r_even, hw_scale);                                                 \
        sr_convert_pair<(B)>(odd, pr, r_odd, hw_scale);                                                   \
    }
    Philox4 ph;
#pragma unroll
    for (int wi = 0; wi < 4; ++wi) {
        // words 0,1 of the call serve the even octet of the pair, words 2,3 the odd one
        if ((wi & 1) == 0) ph = philox_for_hexadecad(seed, (uint64_t)(group_index * 2 + (wi >> 1)));
        uint32_t even, odd;  // converts driven by the even / odd element's random byte; each of their bytes gets written
        asm("" : "=v"(even), "=v"(odd));
        if ((wi & 1) == 0) { QM_SR_PAIR(0, 0) QM_SR_PAIR(1, 2) QM_SR_PAIR(2, 4) QM_SR_PAIR(3, 6) }
        else { QM_SR_PAIR(0, 8) QM_SR_PAIR(1, 10) QM_SR_PAIR(2, 12) QM_SR_PAIR(3, 14) }
        // low nibbles from `even`, high ones from `odd`, sign bits back (n is negated)
        codes[wi] = (uint32_t)__builtin_amdgcn_bitop3_b32((int)even, (int)odd, 0x0f0f0f0f, 0xe4) ^ 0x88888888u;
    }
#undef QM_SR_PAIR
}

template <int MODE, bool WANT_MASK>
__device__ __forceinline__ void quantize_group_regs(const float (&n)[32], uint64_t seed, int64_t group_index,
                                                    GroupCodes& o) {
    constexpr bool kQuest = (MODE == QUEST_RTN || MODE == QUEST_SR);
    constexpr bool kSR = (MODE == ABSMAX_SR || MODE == QUEST_SR);
    o.keep = 0u;
    if constexpr (kQuest) {
        float sq[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) sq[i] = n[i] * n[i];
        const float ms = tree_sum32(sq) * 0.03125f;
        const float m = tree_sum32(n) * 0.03125f;
        const float mm = m * m;
        float var = ms - mm;
        var = var > 0.0f ? var : 0.0f;
        const float sd = __builtin_sqrtf(var);
        const float gs = kQuestG * sd;
        const float s = gs + 1e-8f;
        int E = (int)((f2u(s) >> 23) & 0xffu) - 127;
        E = E > 127 ? 127 : E;
        o.scale_byte = (uint32_t)(E + 127);
        const float hw_scale = pow2i(E);   // the power of two the convert divides by
        o.deq_scale = hw_scale;
        // |n| < 6 * scale  <=>  |t| < 6
        if constexpr (WANT_MASK) o.keep = clip_mask(n, 6.0f * hw_scale, [](float v) { return v; });
        if constexpr (kSR) sr_codes(n, hw_scale, seed, group_index, [](float v) { return v + 0.0f; }, o.w);   // both zeros: +0
        else if (__builtin_expect(ms < __builtin_inff(), 1)) rtn_codes(n, hw_scale, [](float v) { return below_ties(v); }, o.w);
        else rtn_codes(n, hw_scale, [](float v) { return below_ties_any(v); }, o.w);
    } else {
        float a = 0.0f;
#pragma unroll
        for (int i = 0; i < 32; ++i) a = fmaxf(a, fabsf(n[i]));
        const bool all_zero = (a == 0.0f);
        int k = (int)((f2u(a) >> 23) & 0xffu) - 129;
        k = k < -127 ? -127 : (k > 127 ? 127 : k);
        o.scale_byte = (uint32_t)(k + 127);
        o.deq_scale = scale_pow2(kFourThirds, k);
        const auto finish = [&](auto t_of, float hw_scale) {
            // |t| < 6 with t = RN(g 2^-k / d): evaluated on the quotient h = RN(g / d) against 6 * 2^k
            if constexpr (WANT_MASK) o.keep = all_zero ? 0u : clip_mask(n, 6.0f * hw_scale, t_of);
            if constexpr (kSR) sr_codes(n, hw_scale, seed, group_index, t_of, o.w);
            else rtn_codes(n, hw_scale, [&](float v) { return below_ties(t_of(v)); }, o.w);
        };
        // t = RN(RN(g 2^-k) / d) by definition.  For a group whose maximum is at least 2^-60 this is RN(g / d) scaled by
        // 2^-k inside the convert: the two-operation quotient is exact for |g| >= 2^-100, and a smaller element lies
        // below 2^-38 of the scale, so its code is a zero whose sign is the element's own whatever the quotient's last
        // bit.  A group with a smaller non-zero maximum (where g / d would lose bits to underflow) follows the
        // definition literally, with a true division, and hands the convert an already scaled value.
        if (__builtin_expect(a < 0x1p-60f && !all_zero, 0)) finish([&](float v) { return scale_pow2(v, -k) / kFourThirds + 0.0f; }, 1.0f);
        else finish([](float v) { return div_four_thirds_fast(v); }, pow2i(k));   // zeros of either sign: +0
    }
}

template <typename T>
__device__ __forceinline__ void load_group(const T* __restrict__ p, float (&v)[32]) {
    if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint4 raw = reinterpret_cast<const uint4*>(p)[q];
            const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[q * 8 + 2 * i] = u2f(w[i] << 16);
                v[q * 8 + 2 * i + 1] = u2f(w[i] & 0xffff0000u);
            }
        }
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float4 f = reinterpret_cast<const float4*>(p)[q];
            v[q * 4] = f.x; v[q * 4 + 1] = f.y; v[q * 4 + 2] = f.z; v[q * 4 + 3] = f.w;
        }
    }
}

// The group's values: the hardware's FP4 converts hand out code values two by two, the factor and the bf16 rounding follow in fp32
// (225 issue cycles a group; taking the nibbles apart by hand took 770).
template <typename T>
__device__ __forceinline__ void group_values(const GroupCodes& o, uint4 (&out)[2 * sizeof(T)]) {
    typedef __bf16 v2bf16_ __attribute__((ext_vector_type(2)));
    float v[32];
#pragma unroll
    for (int wi = 0; wi < 4; ++wi) {
        // the converts' byte selector must be a literal
#define QM_DEQ_PAIR(B)                                                                               \
    {                                                                                                \
        const v2f q = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(o.w[wi], 1.0f, (B));                  \
        v[wi * 8 + 2 * (B)] = q.x * o.deq_scale;                                                     \
        v[wi * 8 + 2 * (B) + 1] = q.y * o.deq_scale;                                                 \
    }
        QM_DEQ_PAIR(0) QM_DEQ_PAIR(1) QM_DEQ_PAIR(2) QM_DEQ_PAIR(3)
#undef QM_DEQ_PAIR
    }
#pragma unroll
    for (int q = 0; q < (int)(2 * sizeof(T)); ++q) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (sizeof(T) == 2)
                w[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{v[q * 8 + 2 * i], v[q * 8 + 2 * i + 1]}, v2bf16_));
            else
                w[i] = f2u(v[q * 4 + i]);
        }
        out[q] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}
template <typename T>
__device__ __forceinline__ void store_dequant(T* __restrict__ p, const GroupCodes& o) {
    uint4 w[2 * sizeof(T)];
    group_values<T>(o, w);
#pragma unroll
    for (int q = 0; q < (int)(2 * sizeof(T)); ++q) reinterpret_cast<uint4*>(p)[q] = w[q];
}

struct GroupOut {
    uint4* codes;        // [n_groups]
    uint8_t* scales;     // [n_groups]
    uint32_t* maskbits;  // [n_groups] or null
    void* dequant;       // [n_groups * 32] of T or null
};

// times -hd^-1/2 with the column sign folded in: the negated group, as quantize_group_regs takes it
__device__ __forceinline__ void scale_group(float (&v)[32], float c, uint32_t sign_word) {
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        const float cj = u2f(f2u(-c) ^ (((sign_word >> j) & 1u) << 31));  // wave-uniform: stays in scalar registers
        v[j] = v[j] * cj;
    }
}
// -(x @ H) for one chunk of 32
__device__ __forceinline__ void rotate_group(float (&v)[32], float c, uint32_t sign_word, bool rotate = true) {
    if (rotate) butterfly32(v);  // uniform; without it (c = 1, no signs) the group passes through unchanged
    scale_group(v, c, sign_word);
}

typedef __bf16 v2bf16 __attribute__((ext_vector_type(2)));
// round to bf16 and back (round to nearest even, v_cvt_pk_bf16_f32)
__device__ __forceinline__ void round_pair_to_bf16(float& a, float& b) {
    const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{a, b}, v2bf16));
    a = u2f(w << 16);
    b = u2f(w & 0xffff0000u);
}

// silu of a bf16 value, to be rounded to bf16: the hardware's exponential and reciprocal, which for every one of the 65536
// inputs round to the same bf16 value as silu_fixed (tests/test_gpu_fused.py goes through all of them).  A quarter of
// the denominator keeps its reciprocal a normal number up to 2^128; the last bit on top of it settles the one input
// (5.9375) whose result lies 2^-24 from a tie.  silu_fixed is some 35 instructions, a polynomial and an IEEE division, and
// made the producer 92 us at 16384 x 4096 where its bytes take 61; with these six it was 76 (4096 x 1728: 15.2 -> 10.6).
__device__ __forceinline__ float silu_of_bf16(float x) {
    const float e = __builtin_amdgcn_exp2f(x * -1.44269504088896340736f);
    return (x * 0.25f) * __builtin_amdgcn_rcpf(__builtin_fmaf(e, 0.25f, 0x1.000002p-2f));
}
// silu(up) * gate of a group in bf16, rounded after each operation as bf16 tensors are; the product in `up`
__device__ __forceinline__ void swiglu_group_bf16(float (&up)[32], const float (&gate)[32]) {
#pragma unroll
    for (int i = 0; i < 32; ++i) up[i] = silu_of_bf16(up[i]);
#pragma unroll
    for (int i = 0; i < 32; i += 2) round_pair_to_bf16(up[i], up[i + 1]);
#pragma unroll
    for (int i = 0; i < 32; ++i) up[i] = up[i] * gate[i];
#pragma unroll
    for (int i = 0; i < 32; i += 2) round_pair_to_bf16(up[i], up[i + 1]);
}

}  // namespace

}  // namespace qm
