// quartet_amd/csrc/scale_requests.h on the host: for every operand that it lets through, each request that gemm_rows.hip makes of it is of the operand's bytes.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "scale_requests.h"

int main() {
    int let_through = 0, refused = 0;
    for (int64_t K = 128; K <= 1024; K += 128)
        for (int64_t rows : {1, 15, 16, 17, 64}) {
            const int64_t nk = K / 128, codes = (rows + 15) / 16 * 16 * K / 2, scales = rows * K / 32;
            // scales behind the codes without a gap, at the next 256 bytes, in an array of their own in front of them, far behind them; and a byte off
            for (int64_t at : {codes, (codes + 255) / 256 * 256, -scales - 1024, codes + 4096, codes + 1}) {
                std::vector<uint8_t> memory(2 * (size_t)(codes + scales) + 16384);
                const uint8_t* c = memory.data() + scales + 1024 + (16 - reinterpret_cast<uintptr_t>(memory.data() + scales + 1024) % 16) % 16;
                const uint8_t* s = c + at;
                if (!qm::scale_requests_in_operand(c, s, rows, K)) {
                    ++refused;
                    continue;
                }
                ++let_through;
                for (int64_t row = 0; row < rows; ++row)
                    for (int64_t step = 0; step < nk; ++step) {   // a wave's first step can be any
                        const int64_t from = 4 * (step + 4 <= nk ? step : nk - 4) + row * (K / 32);
                        const uint8_t *first = s + from, *last = first + 16;
                        const bool in_scales = first >= s && last <= s + scales, from_codes = first >= c && last <= s + scales && s - (c + codes) < 256 && s >= c + codes;
                        if (reinterpret_cast<uintptr_t>(first) % 4 || !(in_scales || from_codes)) {
                            std::printf("K %lld rows %lld at %lld: step %lld of row %lld reads outside\n", (long long)K, (long long)rows, (long long)at, (long long)step, (long long)row);
                            return EXIT_FAILURE;
                        }
                    }
            }
        }
    std::printf("%d operands let through, %d refused\n", let_through, refused);
    return let_through > 100 && refused > 40 ? EXIT_SUCCESS : EXIT_FAILURE;
}
