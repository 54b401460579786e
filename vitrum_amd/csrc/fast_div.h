// fast_div.h -- correctly rounded binary32 division by a shared denominator.
//
// Built with correctly rounded division, one a / b costs 11 instructions, of
// which most refine the reciprocal of b.  Where several quotients share b
// (vectors scaled by their largest component, barycentrics), div_by reuses
// one refined reciprocal and each further quotient costs 6.
//
// div_by corrects the quotient twice by its exact remainder (Markstein,
// "IA-64 and Elementary Functions", 2000).  That rounds correctly while no
// remainder and no quotient leaves the normal range: callers check the
// operands with div_den and div_key, keep numerators below 2^80 (most are at
// most as large as their denominator) and divide normally otherwise, so
// every quotient has the same bits as a / b.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vtd {

__device__ __forceinline__ float recip_of(float b) {
  const float y = __builtin_amdgcn_rcpf(b);
  return __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
}
__device__ __forceinline__ float div_by(float a, float b, float y) {
  float q = a * y;
  q = __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
  q = __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
  return __builtin_amdgcn_div_fixupf(q, b, a);  // zeros, with their signs
}
// |x| in [2^-40, 2^40]: a denominator.
__device__ __forceinline__ bool div_den(float x) {
  return (__float_as_uint(x) & 0x7FFFFFFFu) - 0x2B800000u <= 0x53800000u - 0x2B800000u;
}
// Numerators are zero or at least 2^-60 in magnitude when the smallest of
// their keys is at least kDivNum (zero wraps to the largest key).  With a
// denominator below 2^40 the quotient then stays above 2^-100.
constexpr uint32_t kDivNum = (0x21800000u << 1) - 1u;
__device__ __forceinline__ uint32_t div_key(float x) { return (__float_as_uint(x) << 1) - 1u; }

}  // namespace vtd
