// Which blocks of a packed tensor may be widened to six bits (expand.hip).  A job of its own, for the grid of the error
// signal's quantizers in front: its eight loads per thread cost nothing there, where asked again by each of the eight
// widening workgroups of a block they cost 10 us of 12 (4096 x 4096 twice).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qm_jobs.h"
#include "qm_kernels.h"

namespace qm {

namespace {

constexpr int kTop6 = 2, kBias6 = 3;     // E3M2: the largest code, 6 = 1.5 * 2^2, times 2^2 is the largest value used, 1.5 * 2^4
constexpr int kSpan6 = kTop6 + kBias6;   // octaves of row scales below the largest that it holds
constexpr int kZeroGroup = 100;          // the scale byte of an all-zero group (2^-27), and of values about as small

// One workgroup per block of 512 rows and 256 columns: are the scales of 32 rows of a column group too far apart somewhere?
struct SpanJob {
    static constexpr int kLds = 16 * (32 * 8 + 8);
    static constexpr int kWaves = 1;
    E5m2Args a;
    unsigned grid_r, blocks;
    explicit SpanJob(const E5m2Args& args)
        : a(args), grid_r((unsigned)((args.R + 511) / 512)), blocks(args.wide ? grid_r * (unsigned)((args.C + kWideStrip - 1) / kWideStrip) : 0u) {}

    __device__ __forceinline__ void run(unsigned bid) const {
        uint8_t* at = reinterpret_cast<uint8_t*>(job_lds);
        const int tid = threadIdx.x, R = (int)a.R, C = (int)a.C, csteps = (int)(padded_cols(C) / 128);
        const unsigned strip = bid / grid_r, block = bid - strip * grid_r;
        const int r0 = (int)block * 512, panel = (int)strip * 2;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = tid + i * 256;
            uint32_t v[2] = {0u, 0u};   // rows and columns past the end: as all-zero groups
            if (r0 + row < R) {
                const uint32_t* src = reinterpret_cast<const uint32_t*>(a.scales_in + (int64_t)(r0 + row) * csteps * 4 + panel * 4);
                v[0] = src[0];
                if (panel + 1 < csteps) v[1] = src[1];
            }
            *reinterpret_cast<uint2*>(at + row * 8 + (row >> 5) * 8) = make_uint2(v[0], v[1]);
        }
        job_requests_issued();
        __syncthreads();
        // two threads per column group and 32 rows
        const int group = (tid >> 1) & 7, rows32 = tid >> 4, row = rows32 * 32 + (tid & 1) * 16;
        int low = 255, top = 0;
        uint32_t zeros = 0;   // rows that look like all-zero groups
        if (panel * 4 + group < C / 32) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int v = at[(row + i) * 8 + rows32 * 8 + group];
                top = v > top ? v : top;
                if (v > kZeroGroup) low = v < low ? v : low;
                else if (r0 + row + i < R) zeros |= 1u << i;
            }
        }
        top = max(top, __shfl_xor(top, 1, 64));
        low = min(low, __shfl_xor(low, 1, 64));
        bool wide = top > low + kSpan6;
        if (top > kZeroGroup + kSpan6 && zeros)   // seldom: are they?
            for (int i = 0; i < 16; ++i)
                if ((zeros >> i) & 1u) {
                    const uint4 q = *reinterpret_cast<const uint4*>(a.codes_in + tiled_code_offset(r0 + row + i, panel + (group >> 2), csteps) + (group & 3) * 16);
                    wide |= ((q.x | q.y | q.z | q.w) & 0x77777777u) != 0;
                }
        const bool any = __syncthreads_or(wide);
        if (tid == 0) a.wide[bid] = any ? 1 : 0;   // [strip][block]
    }
};

}  // namespace

}  // namespace qm
