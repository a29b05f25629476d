// row_terms.h — a row's merged softmax statistics and the loss terms formed
// from them. Device code shared by rowpass.hip and slot.hip.
#pragma once

#include <math.h>

#include "kl_sums.h"

namespace orda {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// Per-row constants: precise logf / IEEE division, or with fast_math the
// hardware approximations (v_log_f32 times ln 2, v_rcp_f32 then a multiply).
__device__ __forceinline__ float rlog(float x, bool fast) {
  return fast ? __builtin_amdgcn_logf(x) * kLn2 : logf(x);
}
__device__ __forceinline__ float rlog2(float x, bool fast) {
  return fast ? __builtin_amdgcn_logf(x) : log2f(x);
}
__device__ __forceinline__ float rdiv(float a, float b, bool fast) {
  return fast ? a * __builtin_amdgcn_rcpf(b) : a / b;
}

struct Stat {
  float m, d1, dT, sx;
};

// KL_row (without T²) of a row pair from its merged statistics s, t and the
// paired GEMM's merged KL sums x (kl_sums.h): the mean of the centred
// difference under p_t^T plus log1p(x.y / t.dT) = lse_s^T - lse_t^T (with
// the shift between the two maxima taken out of both). Precise log1p and
// division of the sums in every profile (they carry the small-KL
// precision; one per row). Should x.y / t.dT not lie in (least, inf), the two
// rows' own sums instead: where s.dT was summed by itself, least = -1/2, below
// which x.y has lost what a student's sum under half the teacher's is (a peaked
// row beside a flat one: off by 1e-5 to 2e-3 of the KL at V = 4096 to 131072).
__device__ __forceinline__ float kl_paired(float2 x, const Stat& s, const Stat& t, float inv_t,
                                           bool fast, float least = -1.f) {
  const float z = x.y / t.dT;
  const float lr = isfinite(z) && z > least ? log1pf(z) : rlog(rdiv(s.dT, t.dT, fast), fast);
  return rdiv(x.x, t.dT, fast) * (kLn2 * inv_t) + lr;
}

// nll of cross_entropy.rs:46-56 from merged stats, in f64.
__device__ __forceinline__ double row_nll(const Stat& s, float xy, double alpha, int64_t v) {
  const double lse = static_cast<double>(s.m) + log(static_cast<double>(s.d1));
  if (alpha > 0.0)
    return lse - (1.0 - alpha) * static_cast<double>(xy) -
           (alpha / static_cast<double>(v)) * static_cast<double>(s.sx);
  return lse - static_cast<double>(xy);
}

}  // namespace orda
