// The six plane products of split3.h on the host: finite values are h + m + l
// exactly, and products of infinities, NaN and zeros are what fp32 gives.
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <stdint.h>

// Host stand-ins for what the header takes from the device compiler.
#define __device__
#define __forceinline__ inline
static float __uint_as_float(uint32_t u) {
  float f;
  memcpy(&f, &u, 4);
  return f;
}
static uint32_t __float_as_uint(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return u;
}
// float -> bf16, to nearest even: the compiler's call for it where the host
// has no instruction.
extern "C" __bf16 __truncsfbf2(float f) {
  uint32_t u = __float_as_uint(f);
  const uint16_t b = static_cast<uint16_t>((u & 0x7fffffffu) > 0x7f800000u ? (u >> 16) | 0x40
                                                                          : (u + 0x7fffu + ((u >> 16) & 1)) >> 16);
  return __builtin_bit_cast(__bf16, b);
}

#include "split3.h"

static float bf16(float f) { return static_cast<float>(static_cast<__bf16>(f)); }

static float planes(float a, float b) {
  float ha, ma, la, hb, mb, lb;
  orda::split3(a, ha, ma, la);
  orda::split3(b, hb, mb, lb);
  la = bf16(la);
  lb = bf16(lb);
  float s = 0.f;
  for (float p : {ha * lb, ha * mb, ma * mb, ma * hb, ha * hb, la * hb}) s += p;
  return s;
}

static bool same(float a, float b) { return a == b || (a != a && b != b); }

int main() {
  uint32_t state = 12345;
  int bad = 0;
  for (int i = 0; i < 1000000; ++i) {
    state = state * 1664525u + 1013904223u;
    const float x = __uint_as_float(state);
    if (!(fabsf(x) <= FLT_MAX) || fabsf(x) < 0x1p-109f) continue;
    float h, m, l;
    orda::split3(x, h, m, l);
    if (h + (m + bf16(l)) != x) ++bad;
  }
  const float inf = INFINITY;
  const float vals[] = {0.f, -0.f, 1.f, -1.f, 1.0038986f, -1.0038986f, 3.e38f, -3.e38f, FLT_MAX, -FLT_MAX,
                        1.e-30f, -1.e-30f, inf, -inf, NAN};
  for (float a : {inf, -inf, NAN, 0.f})
    for (float b : vals) {
      if (same(planes(a, b), a * b) && same(planes(b, a), b * a)) continue;
      printf("%g * %g: planes %g and %g, fp32 %g\n", a, b, planes(a, b), planes(b, a), a * b);
      ++bad;
    }
  printf("%d wrong\n", bad);
  return bad != 0;
}
