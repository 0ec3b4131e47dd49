// Memory helpers of the HIP kernels: typed global pointers, wavefront LDS order.
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

// Orders this wavefront's LDS writes before its later LDS reads by other
// lanes.  The fences name LDS only: a fence on all memory would also wait for
// every global store in flight (loads and stores share one counter here).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

}  // namespace pbbs
