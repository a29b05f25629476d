// slot.hip — the chunk-launcher slot (src/cuda/launch.rs:51-158) on gfx950:
// KL and CE losses and gradients of prepared logits, to separate outputs.
//
// Bound by HBM (fp32 logits: 16 bytes read and 12 written per student/teacher
// logit pair, bf16: 8 and 12). Two kinds of block:
//   * statistics, one block per (row pair, 4096-column segment): both rows'
//     segments are held in registers, so that the maxima, the exponential sums
//     and the KL sums (kl_sums.h) take one read. 8192-column segments measured
//     15 % slower on bf16 logits (fewer blocks in flight), 2048 10 %. Where a
//     fixed scratch does not hold a row's segments (1.75 MiB: V > 94e6) a block
//     takes several times 4096 columns in turn (WIDE);
//   * gradients, elementwise over (row pair, 2048-column block): each wave
//     merges the row's segments while its logits are in flight, the block of
//     column 0 also writes the row's losses.
// Launch k runs the gradients of band k - 1 beside the statistics of band k
// (slot_kernel): 7 % faster on bf16 logits than a launch for each. The bands
// (kBandBytes of logits) do not fit the MALL beside what the gradients write:
// bands of 64 MB measured 380 us at 512 x 131072 fp32, 32 MB 444 (a launch's
// end costs 8 us), 128 MB 353, all rows at once 363.
// Rows start at any address: vectors of four columns begin where the student
// CE output is 16-byte aligned, loads and the other stores take what alignment
// there is (global memory accesses need none on this part). Stores are
// non-temporal where every store instruction covers whole lines (without: 406
// against 353 us); where they do not, non-temporal ones are slower.
// Per call, against a statistics launch for each half with two reads of a row
// and a row-per-workgroup pass taking single elements of unaligned rows: fp32
// 512 x 131072 463 -> 352 us, 300 x 50257 229 -> 110; bf16 512 x 131072 403
// -> 268, 1024 x 32000 218 -> 157, 100 x 50257 182 -> 66.
#include <math.h>

#include "orda_kernels.h"
#include "row_terms.h"

namespace orda {
namespace {

constexpr int kThreads = 256;
constexpr int kSegPer = 16;                    // columns per thread and row
constexpr int kSegCols = kThreads * kSegPer;   // 4096
constexpr int kGradVecs = 2;                   // 4-column vectors per thread and row
constexpr int kGradCols = kThreads * 4 * kGradVecs;
constexpr int64_t kBandBytes = int64_t{128} << 20;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t u16x4u __attribute__((ext_vector_type(4), aligned(2)));

__device__ __forceinline__ void load4(const float* p, float (&x)[4]) {
  const f32x4u w = *reinterpret_cast<const f32x4u*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = w[i];
}
__device__ __forceinline__ void load4(const __bf16* p, float (&x)[4]) {
  const u16x4u w = *reinterpret_cast<const u16x4u*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = __uint_as_float(static_cast<uint32_t>(w[i]) << 16);
}

// The statistics of one row pair's segment: both rows' {max, Σe^(x-max),
// Σe^((x-max)/T), Σx} and the KL sums x, y relative to the two maxima.
struct SegStats {
  float4 s, t;
  float2 c;
};

// An exponential sum relative to a larger maximum m than its own, k = log2(e) / T.
// The maximum skips NaN: a range without another value has -inf beside sums of
// NaN, which times 0 stay NaN, while those of a range that is -inf throughout
// are 0.
__device__ __forceinline__ float shrink(float sum, float own, float m, float k) {
  return sum * (own == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((own - m) * k));
}
// A statistic's two exponential sums relative to a larger maximum.
__device__ __forceinline__ float2 rescale(float4 v, float m, float it2) {
  return make_float2(shrink(v.y, v.x, m, kLog2e), shrink(v.z, v.x, m, it2));
}
// KL sums of a range relative to larger maxima (kl_rebase); a range in which
// one row is -inf throughout keeps what its elements gave (inf or NaN).
__device__ __forceinline__ float2 rebase(float2 c, float4 s, float4 t, float Ms, float Mt, float inv_t) {
  if (s.x != -INFINITY && t.x != -INFINITY) return kl_rebase(c, s.x, t.x, s.z, t.z, Ms, Mt, inv_t);
  const float it2 = inv_t * kLog2e;
  return make_float2(c.x, shrink(s.z, s.x, Ms, it2) - shrink(t.z, t.x, Mt, it2));
}

// The statistics of the kSegCols columns of row pair r from c0 on, in thread 0.
template <typename LT>
__device__ __forceinline__ SegStats col_stats(const SlotArgs& a, int64_t r, int64_t c0) {
  __shared__ float red[kThreads / 64][8];
  const int tid = threadIdx.x;
  const bool teacher = a.kl || a.teacher_ce;
  const LT* srow = static_cast<const LT*>(a.student) + r * a.ld + c0;
  const LT* trow = static_cast<const LT*>(a.teacher) + r * a.ld + c0;
  const int n = static_cast<int>(a.v - c0 < kSegCols ? a.v - c0 : kSegCols);
  float xs[kSegPer], xt[kSegPer];
  auto load = [&](const LT* row, float (&x)[kSegPer]) {
#pragma unroll
    for (int q = 0; q < kSegPer / 4; ++q) {
      const int j = (q * kThreads + tid) * 4;
      float w[4];
      if (j + 4 <= n) {
        load4(row + j, w);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = j + i < n ? static_cast<float>(row[j + i]) : -INFINITY;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) x[4 * q + i] = w[i];
    }
  };
  load(srow, xs);
  if (teacher) load(trow, xt);
  // maxima over the block
  float ms = -INFINITY, mt = -INFINITY;
#pragma unroll
  for (int k = 0; k < kSegPer; ++k) {
    ms = fmaxf(ms, xs[k]);
    if (teacher) mt = fmaxf(mt, xt[k]);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    ms = fmaxf(ms, __shfl_xor(ms, o));
    mt = fmaxf(mt, __shfl_xor(mt, o));
  }
  if ((tid & 63) == 0) {
    red[tid >> 6][0] = ms;
    red[tid >> 6][1] = mt;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) {
    ms = fmaxf(ms, red[w][0]);
    mt = fmaxf(mt, red[w][1]);
  }
  __syncthreads();
  // Sums relative to the maxima (relative to 0 where a row is all -inf, so
  // that its terms are e^-inf = 0).
  const float os = ms == -INFINITY ? 0.f : -ms * kLog2e, ot = mt == -INFINITY ? 0.f : -mt * kLog2e;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // d1s, sxs, d1t, dTt, sxt, cross, diff, dTs
#pragma unroll
  for (int q = 0; q < kSegPer / 4; ++q) {
    const bool whole = (q * kThreads + tid) * 4 + 4 <= n;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!whole && (q * kThreads + tid) * 4 + i >= n) continue;
      const float s = xs[4 * q + i];
      const float ts = fmaf(s, kLog2e, os);   // explicit: equal rows give equal terms
      const float aTs = __builtin_amdgcn_exp2f(ts * a.inv_t);
      v[0] += __builtin_amdgcn_exp2f(ts);
      v[1] += s;
      if (teacher) {
        const float t = xt[4 * q + i];
        const float tt = fmaf(t, kLog2e, ot);
        const float aTt = __builtin_amdgcn_exp2f(tt * a.inv_t);
        v[2] += __builtin_amdgcn_exp2f(tt);
        v[3] += aTt;
        v[4] += t;
        v[5] = fmaf(aTt, tt - ts, v[5]);
        v[6] += aTs - aTt;
      }
      v[7] += aTs;   // by itself: out of v[6] + v[3] it would lose a sum small beside the teacher's
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v[k] += __shfl_xor(v[k], o);
    if ((tid & 63) == 0) red[tid >> 6][k] = v[k];
  }
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      v[k] = red[0][k];
#pragma unroll
      for (int w = 1; w < kThreads / 64; ++w) v[k] += red[w][k];
    }
  }
  return {make_float4(ms, v[0], v[7], v[1]), make_float4(mt, v[2], v[3], v[4]), make_float2(v[5], v[6])};
}

// Two ranges' statistics as one's.
__device__ __forceinline__ SegStats join(const SegStats& a, const SegStats& b, float inv_t) {
  const float it2 = inv_t * kLog2e, ms = fmaxf(a.s.x, b.s.x), mt = fmaxf(a.t.x, b.t.x);
  const float2 sa = rescale(a.s, ms, it2), sb = rescale(b.s, ms, it2);
  const float2 ta = rescale(a.t, mt, it2), tb = rescale(b.t, mt, it2);
  const float2 ca = rebase(a.c, a.s, a.t, ms, mt, inv_t), cb = rebase(b.c, b.s, b.t, ms, mt, inv_t);
  return {make_float4(ms, sa.x + sb.x, sa.y + sb.y, a.s.w + b.s.w),
          make_float4(mt, ta.x + tb.x, ta.y + tb.y, a.t.w + b.t.w), make_float2(ca.x + cb.x, ca.y + cb.y)};
}

// Segment sg: kSegCols columns, or WIDE, a.seg_cols of them in turn.
template <typename LT, bool WIDE>
__device__ __forceinline__ void slot_stats(const SlotArgs& a, int64_t r, int64_t sg, SegStats* out) {
  const int64_t c0 = sg * (WIDE ? a.seg_cols : kSegCols);
  SegStats st = col_stats<LT>(a, r, c0);
  if constexpr (WIDE) {
    const int64_t end = c0 + a.seg_cols < a.v ? c0 + a.seg_cols : a.v;
    for (int64_t c = c0 + kSegCols; c < end; c += kSegCols) {
      __syncthreads();   // thread 0 has read the last columns' sums
      st = join(st, col_stats<LT>(a, r, c), a.inv_t);
    }
  }
  if (threadIdx.x == 0) out[sg] = st;
}

template <typename LT>
__device__ __forceinline__ void slot_grad(const SlotArgs& a, int64_t r, int64_t ci, int64_t nseg,
                                          const SegStats* st) {
  const int tid = threadIdx.x, lane = tid & 63;
  const bool kl = a.kl, tg = a.teacher_ce, teacher = kl || tg;
  const int64_t v = a.v;
  const LT* srow = static_cast<const LT*>(a.student) + r * a.ld;
  const LT* trow = static_cast<const LT*>(a.teacher) + r * a.ld;
  float* gk = a.grad_kl + r * v;
  float* gs = a.grad_ce + r * v;
  float* gt = a.grad_ce + (a.n_rows + r) * v;
  // Vectors start `off` columns past a multiple of the block: the first column
  // at which the student's CE output is 16-byte aligned. The block of column
  // 0 takes the columns before it, one a thread, as a last, short vector.
  const int off = static_cast<int>((16 - (reinterpret_cast<uintptr_t>(gs) & 15)) >> 2) & 3;
  const bool lines = a.out_lines;   // every store instruction covers whole lines
  int64_t col[kGradVecs];
  int cnt[kGradVecs];
  float xs[kGradVecs][4], xt[kGradVecs][4] = {};
#pragma unroll
  for (int q = 0; q < kGradVecs; ++q) {
    const int64_t j = ci * kGradCols + (q * kThreads + tid) * 4 + off;
    col[q] = j;
    cnt[q] = static_cast<int>(j + 4 <= v ? 4 : j < v ? v - j : 0);
    if (cnt[q] == 4) {
      load4(srow + j, xs[q]);
      if (teacher) load4(trow + j, xt[q]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xs[q][i] = i < cnt[q] ? static_cast<float>(srow[j + i]) : 0.f;
        if (teacher) xt[q][i] = i < cnt[q] ? static_cast<float>(trow[j + i]) : 0.f;
      }
    }
  }
  // the row's statistics from its segments, in every wave
  const float inv_t = a.inv_t, it2 = inv_t * kLog2e;
  const float4 none = make_float4(-INFINITY, 0.f, 0.f, 0.f);
  Stat ss{-INFINITY, 0.f, 0.f, 0.f}, tt{-INFINITY, 0.f, 0.f, 0.f};
  for (int64_t k = lane; k < nseg; k += 64) {
    ss.m = fmaxf(ss.m, st[k].s.x);
    tt.m = fmaxf(tt.m, st[k].t.x);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    ss.m = fmaxf(ss.m, __shfl_xor(ss.m, o));
    tt.m = fmaxf(tt.m, __shfl_xor(tt.m, o));
  }
  float2 xc = make_float2(0.f, 0.f);
  for (int64_t k = lane; k < nseg; k += 64) {
    const float4 s = st[k].s, t = teacher ? st[k].t : none;
    const float2 ds = rescale(s, ss.m, it2), dt = rescale(t, tt.m, it2);
    ss.d1 += ds.x;
    ss.dT += ds.y;
    ss.sx += s.w;
    tt.d1 += dt.x;
    tt.dT += dt.y;
    tt.sx += t.w;
    if (kl && ci == 0) {
      const float2 c = rebase(st[k].c, s, t, ss.m, tt.m, inv_t);
      xc.x += c.x;
      xc.y += c.y;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    ss.d1 += __shfl_xor(ss.d1, o);
    ss.dT += __shfl_xor(ss.dT, o);
    tt.d1 += __shfl_xor(tt.d1, o);
    tt.dT += __shfl_xor(tt.dT, o);
    if (ci == 0) {
      ss.sx += __shfl_xor(ss.sx, o);
      tt.sx += __shfl_xor(tt.sx, o);
      xc.x += __shfl_xor(xc.x, o);
      xc.y += __shfl_xor(xc.y, o);
    }
  }
  const int32_t y = a.targets[r];
  // A target outside [0, V) that is not ignore_index counts as ignored.
  const bool ignored = y == a.ignore_index || y < 0 || y >= v;
  const float o1s = (ss.m + logf(ss.d1)) * kLog2e, oTs = (ss.m * inv_t + logf(ss.dT)) * kLog2e;
  const float o1t = (tt.m + logf(tt.d1)) * kLog2e, oTt = (tt.m * inv_t + logf(tt.dT)) * kLog2e;
  const double alpha = static_cast<double>(a.label_smoothing);
  const float eps = static_cast<float>(alpha / static_cast<double>(v));
  const float one_m_a = 1.0f - a.label_smoothing;
  const float ws = ignored ? 0.f : a.w_s, wt = ignored ? 0.f : a.w_t;   // cross_entropy.rs:59
  const float gsc = ignored ? 0.f : a.kl_grad_scale;                    // kl.rs:85
  auto elem = [&](int64_t j, float x, float z, float& g, float& k, float& t) {
    float prob = __builtin_amdgcn_exp2f(fmaf(x, kLog2e, -o1s)) - eps;
    if (j == y) prob -= one_m_a;
    g = prob * ws;
    k = kl ? gsc * (__builtin_amdgcn_exp2f(fmaf(x, it2, -oTs)) - __builtin_amdgcn_exp2f(fmaf(z, it2, -oTt)))
           : 0.f;
    t = 0.f;
    if (tg) {
      float pr = __builtin_amdgcn_exp2f(fmaf(z, kLog2e, -o1t)) - eps;
      if (j == y) pr -= one_m_a;
      t = pr * wt;
    }
  };
  const bool kvec = ((reinterpret_cast<uintptr_t>(gk) ^ reinterpret_cast<uintptr_t>(gs)) & 15) == 0;
#pragma unroll
  for (int q = 0; q < kGradVecs; ++q) {
    const int64_t j = col[q];
    f32x4 g, k, t;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float e0, e1, e2;
      elem(j + i, xs[q][i], xt[q][i], e0, e1, e2);
      g[i] = e0;
      k[i] = e1;
      t[i] = e2;
    }
    if (cnt[q] == 4 && lines) {
      __builtin_nontemporal_store(g, reinterpret_cast<f32x4*>(gs + j));
      __builtin_nontemporal_store(k, reinterpret_cast<f32x4*>(gk + j));
      if (tg) __builtin_nontemporal_store(t, reinterpret_cast<f32x4*>(gt + j));
    } else if (cnt[q] == 4) {
      *reinterpret_cast<f32x4*>(gs + j) = g;
      if (kvec) *reinterpret_cast<f32x4*>(gk + j) = k;
      else *reinterpret_cast<f32x4u*>(gk + j) = k;
      if (tg) *reinterpret_cast<f32x4u*>(gt + j) = t;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i >= cnt[q]) continue;
        gs[j + i] = g[i];
        gk[j + i] = k[i];
        if (tg) gt[j + i] = t[i];
      }
    }
  }
  if (ci != 0) return;
  if (tid < off && tid < v) {   // the columns before the first vector
    float g, k, t;
    elem(tid, static_cast<float>(srow[tid]), teacher ? static_cast<float>(trow[tid]) : 0.f, g, k, t);
    gs[tid] = g;
    gk[tid] = k;
    if (tg) gt[tid] = t;
  }
  if (tid == 0) {
    a.ce_loss[r] = ignored ? 0.f : static_cast<float>(row_nll(ss, static_cast<float>(srow[y]), alpha, v));
    if (tg)
      a.ce_loss[a.n_rows + r] =
          ignored ? 0.f : static_cast<float>(row_nll(tt, static_cast<float>(trow[y]), alpha, v));
    a.kl_row[r] = kl && !ignored ? kl_paired(xc, ss, tt, inv_t, false, -0.5f) * a.t_sq : 0.f;
  }
}

// Launch k of a call: the gradients of band k - 1 beside the statistics of
// band k, row by row, so that reads and writes run together and a launch's
// last blocks are of both kinds. Bands use the two halves of the scratch in
// turn.
template <typename LT, bool WIDE>
__global__ __launch_bounds__(kThreads) void slot_kernel(SlotArgs a, int64_t k, int64_t band, int64_t nseg,
                                                        int64_t chunks, int64_t per) {
  const int64_t row = blockIdx.x / per;
  int64_t i = blockIdx.x - row * per;
  // the first launch has no gradients, the last no statistics
  const bool grads = k > 0 && i < chunks;
  if (k > 0 && !grads) i -= chunks;
  const int64_t r = (grads ? k - 1 : k) * band + row;
  if (row >= band || r >= a.n_rows) return;
  SegStats* half = static_cast<SegStats*>(a.scratch) + (((grads ? k - 1 : k) & 1) * band + row) * nseg;
  if (grads) slot_grad<LT>(a, r, i, nseg, half);
  else slot_stats<LT, WIDE>(a, r, i, half);
}

int64_t segments(int64_t v, int64_t cols) { return (v + cols - 1) / cols; }

}  // namespace

int64_t slot_band_rows(DType t, int64_t n_rows, int64_t v) {
  const int64_t b = kBandBytes / (2 * v * dtype_size(t));
  return b < 1 ? 1 : b < n_rows ? b : n_rows;
}

int64_t slot_seg_cols(int64_t v, int64_t scratch) {
  const int64_t most = scratch / (2 * static_cast<int64_t>(sizeof(SegStats)));
  return (segments(v, kSegCols) + most - 1) / most * kSegCols;
}

int64_t slot_scratch_bytes(int64_t band, int64_t v, int64_t seg_cols) {
  return 2 * band * segments(v, seg_cols) * static_cast<int64_t>(sizeof(SegStats));
}

hipError_t launch_slot(const SlotArgs& a, int64_t band, hipStream_t s) {
  if (a.n_rows <= 0) return hipSuccess;
  const int64_t nseg = segments(a.v, a.seg_cols);
  const int64_t chunks = (a.v + kGradCols - 1) / kGradCols;
  const int64_t bands = (a.n_rows + band - 1) / band;
  if (band < 1 || band * (nseg + chunks) > 0x7fffffff || a.seg_cols < 1 || a.seg_cols % kSegCols)
    return hipErrorInvalidValue;
  using K = void (*)(SlotArgs, int64_t, int64_t, int64_t, int64_t, int64_t);
  const bool wide = a.seg_cols > kSegCols, bf16 = a.ltype == DType::BF16;
  const K kernel = bf16 ? (wide ? K(slot_kernel<__bf16, true>) : K(slot_kernel<__bf16, false>))
                        : (wide ? K(slot_kernel<float, true>) : K(slot_kernel<float, false>));
  for (int64_t k = 0; k <= bands; ++k) {
    const int64_t per = (k > 0 ? chunks : 0) + (k < bands ? nseg : 0);
    const int64_t left = a.n_rows - (k > 0 ? k - 1 : 0) * band;
    const dim3 grid(static_cast<unsigned>((left < band ? left : band) * per));
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, s, a, k, band, nseg, chunks, per);
  }
  return hipGetLastError();
}

}  // namespace orda
