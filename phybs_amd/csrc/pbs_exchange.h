// pbs_exchange.h -- values passed between the workgroups of a resident (cooperative) kernel.
//
// They cross as relaxed atomics at agent scope (8 or 4 bytes each, written through to and read from
// the point where all XCDs see them), and they are their own flags: an entry holds all-ones bits until
// its owner has written it, a reader polls until it does not (a computed value with that bit
// pattern, a NaN, is replaced by another NaN).  Every poll is bounded.
#pragma once
#include <hip/hip_runtime.h>

namespace pbs {

template <typename R> struct Bits;
template <> struct Bits<double> {
  typedef unsigned long long type;
  static constexpr type none = ~0ULL, nan = 0x7ff8000000000000ULL;
};
template <> struct Bits<float> {
  typedef unsigned type;
  static constexpr type none = ~0U, nan = 0x7fc00000U;
};
template <typename R> __device__ __forceinline__ void publish(R *p, R v) {
  typedef typename Bits<R>::type B;
  B b = __builtin_bit_cast(B, v);
  if (b == Bits<R>::none) b = Bits<R>::nan;
  __hip_atomic_store((B *)p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename R> __device__ __forceinline__ void clear(R *p) {
  __hip_atomic_store((typename Bits<R>::type *)p, Bits<R>::none, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename R> __device__ __forceinline__ typename Bits<R>::type poll(const R *p) {
  return __hip_atomic_load((const typename Bits<R>::type *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// One more poll in vain: whether to give up (after `polls` of them, or when another has).
__device__ __forceinline__ bool give_up(int &spin, int polls, int *abort) {
  return ++spin >= polls || (spin % 1024 == 0 && __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

}  // namespace pbs
