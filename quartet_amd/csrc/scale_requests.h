// Where a request for four K steps of a row's scales (gemm_rows.hip) reads.  No HIP in here: tests/scale_requests_check.cpp runs it on the host.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace qm {

// Bytes that the requests of an operand of K indices a row (a multiple of 128, four bytes of scales to each 128) read in front of its scales: they are
// sixteen bytes and end with the row's last byte at the latest.
inline int64_t bytes_before_scales(int64_t K) { return K >= 512 ? 0 : 16 - K / 32; }

// Whether they read nothing that is not the operand's: rows of four steps and more, or scales that lie behind the operand's codes, a packed operand's distance
// (to the next multiple of 256 bytes) at most; and whether they are aligned.
inline bool scale_requests_in_operand(const uint8_t* codes, const uint8_t* scales, int64_t rows, int64_t K) {
    if (reinterpret_cast<uintptr_t>(scales) % 4) return false;
    if (bytes_before_scales(K) == 0) return true;
    const uintptr_t end = reinterpret_cast<uintptr_t>(codes) + (uintptr_t)((rows + 15) / 16 * 16 * (K / 2)), at = reinterpret_cast<uintptr_t>(scales);
    return at >= end && at - end < 256;
}

}  // namespace qm
