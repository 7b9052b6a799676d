// Device pieces shared by the proposal's inference and training kernels: bf16 conversion, the MFMA
// fragment, and the input encoding.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mlp.hpp"

namespace gprt {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

union Frag {
  bf16x8_t v;
  uint4 u;
  uint16_t h[8];
};

__device__ __forceinline__ f32x4_t mfma16(const Frag &a, const Frag &b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}

// FP32 -> bf16 with round-to-nearest-even (NaN stays NaN).
__host__ __device__ __forceinline__ uint16_t f2bf(float f) {
  union {
    float f;
    uint32_t u;
  } x;
  x.f = f;
  if ((x.u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((x.u >> 16) | 0x40u);
  const uint32_t r = 0x7FFFu + ((x.u >> 16) & 1u);
  return (uint16_t)((x.u + r) >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ uint32_t pack2(float lo, float hi) { return (uint32_t)f2bf(lo) | ((uint32_t)f2bf(hi) << 16); }

}  // namespace gprt
