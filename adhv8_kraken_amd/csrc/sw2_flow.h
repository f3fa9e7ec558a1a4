// Words handed from one workgroup of a kernel to another while both run: a word
// holds EMPTY until it is stored, by an agent-scope store (past the XCDs'
// private L2s), and readers poll the word itself, so a hand-over is one store
// and one load deep and needs no fence.
#pragma once
#include <hip/hip_runtime.h>

namespace sw2 {

// EMPTY is a NaN no arithmetic produces.
template <typename T>
struct Slot;
template <>
struct Slot<double> {
    using U = unsigned long long;
    static constexpr U EMPTY = 0xfff8dead0badf00dull, QNAN = 0x7ff8000000000000ull;
};
template <>
struct Slot<float> {
    using U = unsigned;
    static constexpr U EMPTY = 0xffdeadadu, QNAN = 0x7fc00000u;
};

template <typename T>
__device__ __forceinline__ typename Slot<T>::U peek(const T *p) {
    return __hip_atomic_load((const typename Slot<T>::U *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void put_raw(T *p, typename Slot<T>::U u) {
    __hip_atomic_store((typename Slot<T>::U *)p, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void put(T *p, T v) {
    typename Slot<T>::U u = __builtin_bit_cast(typename Slot<T>::U, v);
    if (u == Slot<T>::EMPTY) u = Slot<T>::QNAN;
    put_raw(p, u);
}

}  // namespace sw2
