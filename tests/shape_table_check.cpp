// quartet_amd/csrc/shape_table.h on the host: shapes that a program asks for in turn are worked out once each.
#include <cstdio>
#include <cstdlib>

#include "shape_table.h"

struct Entry {
    int64_t M = -1, N = 0, K = 0;
    int flags = -1;
    int64_t value = 0;
};

int main() {
    // the products of twelve layers (forward, both gradients, with and without a cut) at one token count after the other
    const int64_t layers[][2] = {{640, 1920}, {640, 640}, {640, 3456}, {1728, 640}, {1536, 4608}, {1536, 1536}, {1536, 8192}, {4096, 1536},
                                 {4096, 4096}, {4096, 11008}, {11008, 4096}, {4096, 22016}};
    int64_t worst = 0, total = 0, shapes = 0;
    for (int64_t T : {64, 512, 1000, 4096, 8192, 16480, 16384, 32768}) {
        qm::ShapeTable<Entry, 6> table;
        int64_t made = 0, asked = 0;
        for (int step = 0; step < 100; ++step)
            for (const auto& l : layers) {
                const int64_t I = l[0], O = l[1], ask[3][3] = {{T, O, I}, {T, I, O}, {O, I, T}};
                for (int flags = 2; flags < 4; ++flags)
                    for (const auto& s : ask) {
                        const auto make = [&] { ++made; return Entry{s[0], s[1], s[2], flags, s[0] * 3 + s[1] * 5 + s[2] * 7 + flags}; };
                        if (table.find(s[0], s[1], s[2], flags, make).value != s[0] * 3 + s[1] * 5 + s[2] * 7 + flags) return std::puts("wrong entry"), 1;
                        ++asked;
                    }
            }
        total += made; shapes += 72;
        if (made > worst) worst = made;
        if (made * 10 > asked) return std::printf("T %lld: %lld of %lld worked out anew\n", (long long)T, (long long)made, (long long)asked), 1;
    }
    // one layer by itself: never more than once per shape
    for (const auto& l : layers) {
        qm::ShapeTable<Entry, 6> table;
        int made = 0;
        for (int step = 0; step < 50; ++step)
            for (int64_t K : {(int64_t)512, l[1]}) {
                const int64_t M = K == 512 ? l[1] : 512, N = l[0];
                table.find(M, N, K, 3, [&] { ++made; return Entry{M, N, K, 3, 0}; });
            }
        if (made != 2) return std::printf("%lld x %lld: %d\n", (long long)l[0], (long long)l[1], made), 1;
    }
    std::printf("shapes %lld worked out %lld ok\n", (long long)shapes, (long long)total);
    return 0;
}
