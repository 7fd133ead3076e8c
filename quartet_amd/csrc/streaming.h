// Loads and stores past the caches: they displace nothing that others keep there, and what they store is not there for a reader.
// Whether that pays, and from which size on, is measured kernel by kernel (each says so beside its accesses).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qm {

// A tensor of this size and a result as large are most of what the memory-side cache holds (256 MB).  Kernels that gain only on tensors
// which do not stay there take these accesses from here on.
constexpr int64_t kPastTheCaches = 96ll << 20;
// A result from here on cannot be there as a whole when the next launch reads it.
constexpr int64_t kMoreThanTheCaches = 256ll << 20;

template <typename V>
__device__ __forceinline__ V stream_load(const V* p) {
    static_assert(sizeof(V) == 8 || sizeof(V) == 16, "whole vectors");
    typedef uint32_t raw __attribute__((ext_vector_type(sizeof(V) / 4)));
    return __builtin_bit_cast(V, __builtin_nontemporal_load(reinterpret_cast<const raw*>(p)));
}
template <typename V>
__device__ __forceinline__ void stream_store(V* p, const V& v) {
    static_assert(sizeof(V) == 8 || sizeof(V) == 16, "whole vectors");
    typedef uint32_t raw __attribute__((ext_vector_type(sizeof(V) / 4)));
    __builtin_nontemporal_store(__builtin_bit_cast(raw, v), reinterpret_cast<raw*>(p));
}

}  // namespace qm
