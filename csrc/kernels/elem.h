// One-element and four-element access of the two projection types (bf16, and fp32 for the engine
// that computes everything in 32-bit), shared by the kernels that are templates over the type.
#pragma once
#include "common.h"

LSA_DEVICE float ld1(const float* p) { return *p; }
LSA_DEVICE float ld1(const bf16_raw* p) { return bf2f(*p); }
LSA_DEVICE void st1(float* p, float v) { *p = v; }
LSA_DEVICE void st1(bf16_raw* p, float v) { *p = f2bf(v); }
LSA_DEVICE void st4(float* p, f32x4_t v) { *reinterpret_cast<f32x4_t*>(p) = v; }
LSA_DEVICE void st4(bf16_raw* p, f32x4_t v) {
  const unsigned lo = f2bf2(v[0], v[1]);
  const unsigned hi = f2bf2(v[2], v[3]);
  *reinterpret_cast<u32x2_t*>(p) = u32x2_t{lo, hi};
}

LSA_DEVICE float sigmoid(float z) { return 1.0f / (1.0f + __expf(-z)); }

// the sum of a and that of b over both halves of the wave (of each 32 lanes): a's in the lower one, b's in the upper one
LSA_DEVICE float halves(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
LSA_DEVICE float quarters(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
