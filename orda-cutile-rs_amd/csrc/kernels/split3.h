// split3.h — an fp32 value as the sum of three bf16 values, the operand form
// of the fp32 GEMMs on the bf16 matrix units (gemm.hip).
#pragma once

#include <float.h>
#include <math.h>
#include <stdint.h>

namespace orda {

// h, m, l: x rounded to bf16 (nearest even), then the two remainders likewise.
// Each remainder is exact in fp32 and 24 bits of significand are three times
// eight, so h + m + l == x for every finite x whose last bit is at or above
// the smallest bf16 denormal, 2^-133 (below it l rounds). h truncates where
// rounding would overflow. An infinity or a NaN is l, beside an h of its sign
// and size 1: of the six plane products only l times the other value's h meets
// it, so that infinity times a value is the infinity of the right sign, and
// times another infinity too (1 * inf twice and 1 * 1). As h, it would also meet
// the other value's m and l, of either sign, or zero: a NaN.
__device__ __forceinline__ void split3(float x, float& h, float& m, float& l) {
  const bool finite = fabsf(x) <= FLT_MAX;
  h = static_cast<float>(static_cast<__bf16>(x));
  if (!(fabsf(h) <= FLT_MAX)) h = finite ? __uint_as_float(__float_as_uint(x) & 0xffff0000u) : copysignf(1.f, x);
  const float r = finite ? x - h : 0.f;
  m = static_cast<float>(static_cast<__bf16>(r));
  l = finite ? r - m : x;   // stored rounded to bf16
}

// Two values' planes as packed bf16 pairs, p[0] = h, p[1] = m, p[2] = l.
__device__ __forceinline__ void split3_pack(float a, float b, uint32_t (&p)[3]) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  float ha, ma, la, hb, mb, lb;
  split3(a, ha, ma, la);
  split3(b, hb, mb, lb);
  p[0] = __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(ha), static_cast<__bf16>(hb)});
  p[1] = __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(ma), static_cast<__bf16>(mb)});
  p[2] = __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(la), static_cast<__bf16>(lb)});
}

}  // namespace orda
