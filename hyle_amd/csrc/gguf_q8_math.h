// Device helpers of the GGUF products with 8-bit activation blocks (gguf_matvec_q8.hip, gguf_matvec_strips.hip).
#pragma once

#include "device_common.h"

namespace hyle_hip {
namespace {

// a * b + c for factors that fit 24 signed bits (v_mad_i32_i24; a full 32-bit multiply is four
// times slower)
__device__ __forceinline__ int mad24(int a, int b, int c) { return __mul24(a, b) + c; }

__device__ __forceinline__ int dot4(uint32_t weights, uint32_t codes, int sum) {
  return __builtin_amdgcn_sdot4((int)weights, (int)codes, sum, false);
}

// Block barrier that orders LDS accesses only: the weight loads issued before it stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace
}  // namespace hyle_hip
