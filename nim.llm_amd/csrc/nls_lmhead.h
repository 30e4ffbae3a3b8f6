// nls_lmhead.h -- what the output projection's translation units share.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nls_internal.h"

namespace nls {

__device__ __forceinline__ uint32_t lm_ld_u16(const uint8_t* p) {
  uint16_t v;
  __builtin_memcpy(&v, p, 2);
  return v;
}
__device__ __forceinline__ uint4 lm_ld_16(const void* p) {
  uint4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}
// IEEE half to float: exact for every finite half (subnormals included).
__device__ __forceinline__ float lm_half_f(uint32_t bits) {
  _Float16 h;
  const uint16_t b = (uint16_t)bits;
  __builtin_memcpy(&h, &b, 2);
  return (float)h;
}

// nls_lmbatch.hip: the K formats' int8 path on the matrix cores, after the
// activations are quantised into the workspace.
hipError_t launch_lm_batch(const LmHeadCall& c, hipStream_t s);

}  // namespace nls
