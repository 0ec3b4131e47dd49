// Helpers of the HIP kernels: typed global pointers, wavefront LDS order,
// cross-lane moves and scans.
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

// Cross-lane moves through DPP (a VALU operand modifier, a few cycles)
// instead of ds_bpermute (an LDS round trip).  `old` is what lanes without a
// source lane (or masked rows) receive.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ unsigned dpp_u32(unsigned x, unsigned old) {
  return (unsigned)__builtin_amdgcn_update_dpp((int)old, (int)x, kCtrl, kRowMask, 0xf, false);
}
template <int kCtrl, int kRowMask>
__device__ __forceinline__ int dpp_i32(int x, int old) {
  return __builtin_amdgcn_update_dpp(old, x, kCtrl, kRowMask, 0xf, false);
}
constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118;
constexpr int kRowBcast15 = 0x142, kRowBcast31 = 0x143, kWaveShr1 = 0x138;

// Inclusive sum over the wavefront through DPP.
__device__ __forceinline__ unsigned wave_inclusive_sum_dpp(unsigned x) {
  x += dpp_u32<kRowShr1, 0xf>(x, 0u);
  x += dpp_u32<kRowShr2, 0xf>(x, 0u);
  x += dpp_u32<kRowShr4, 0xf>(x, 0u);
  x += dpp_u32<kRowShr8, 0xf>(x, 0u);
  x += dpp_u32<kRowBcast15, 0xa>(x, 0u);
  x += dpp_u32<kRowBcast31, 0xc>(x, 0u);
  return x;
}

// Inclusive maximum over the wavefront through DPP.
__device__ __forceinline__ unsigned wave_inclusive_max_dpp(unsigned x) {
  x = max(x, dpp_u32<kRowShr1, 0xf>(x, 0u));
  x = max(x, dpp_u32<kRowShr2, 0xf>(x, 0u));
  x = max(x, dpp_u32<kRowShr4, 0xf>(x, 0u));
  x = max(x, dpp_u32<kRowShr8, 0xf>(x, 0u));
  x = max(x, dpp_u32<kRowBcast15, 0xa>(x, 0u));
  x = max(x, dpp_u32<kRowBcast31, 0xc>(x, 0u));
  return x;
}

}  // namespace pbbs
