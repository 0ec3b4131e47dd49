// Typed global-memory pointers for the HIP kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace pbbs {

// Device pointers typed in the global address space, so loads, stores and
// atomics through them compile to global_* instructions.  Generic (flat)
// accesses also count against the LDS counter, so every LDS or cross-lane
// wait would otherwise wait for the outstanding memory loads too.
#define PBBS_GLOBAL __attribute__((address_space(1)))
template <typename T>
using gptr = PBBS_GLOBAL T*;
template <typename T>
__device__ __forceinline__ gptr<T> glob(T* p) {
  return (gptr<T>)p;
}
// Generic pointer for the atomic builtins; the compiler still sees the
// global origin and emits global atomics.
template <typename T>
__device__ __forceinline__ T* gen(gptr<T> p) {
  return (T*)p;
}

}  // namespace pbbs
