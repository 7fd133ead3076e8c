// Loads and stores of values that no launch soon after reads: they pass through the caches without displacing what others keep there.
// Whether that pays is measured kernel by kernel (each says so beside its accesses).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qm {

// Most of what the memory-side cache holds (256 MB).  Kernels that gain only on tensors which do not stay there take these accesses
// from here on.
constexpr int64_t kPastTheCaches = 96ll << 20;

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
