// What the host has worked out for a shape, remembered: a table of fixed size, four entries to a slot, replaced in turn.
#pragma once
#include <stdint.h>

#include <initializer_list>

namespace qm {

// Extents are multiples of 64 and flags small: a slot taken from their low bits would be one and the same for all of them.
// Multiplying by 2^64 / phi spreads them over the high bits (Knuth's multiplicative hashing), which is where it is read.
constexpr uint64_t kGoldenRatio64 = 0x9E3779B97F4A7C15ull;
inline uint64_t shape_hash(int64_t M, int64_t N, int64_t K, int flags) {
    uint64_t h = (uint64_t)M;
    for (const uint64_t v : {(uint64_t)N, (uint64_t)K, (uint64_t)flags}) {
        h *= kGoldenRatio64;
        h = (h ^ (h >> 32)) + v;
    }
    return h * kGoldenRatio64;
}

// Entry: a struct with members M, N, K, flags that are set where the entry holds that shape; default-constructed ones hold none.
template <class Entry, int SLOTS_LOG2>
class ShapeTable {
    struct Slot {
        Entry e[4];
        unsigned next = 0;   // the entry replaced next
    };
    Slot slots_[1 << SLOTS_LOG2];

  public:
    template <class Make>   // make() -> Entry of this shape
    const Entry& find(int64_t M, int64_t N, int64_t K, int flags, const Make& make) {
        Slot& s = slots_[shape_hash(M, N, K, flags) >> (64 - SLOTS_LOG2)];
        for (const Entry& e : s.e)
            if (e.M == M && e.N == N && e.K == K && e.flags == flags) return e;
        return s.e[s.next++ % 4] = make();
    }
};

}  // namespace qm
