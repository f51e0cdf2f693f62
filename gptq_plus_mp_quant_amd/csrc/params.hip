// Quantizer parameters, per-subgroup gathers and the final write-back.
//  - rq_find_params:      WeightQuantizer.find_params, per-channel min/max (utils/quant_utils.py:390-421),
//                         also per static column group (gptq_utils/gptq_plus_utils.py:994-1002) and
//                         find_params_weight_groupwise (utils/quant_utils.py:333-388, clip_zero = 0)
//  - rq_prepare_subgroup: row slice, dead columns, act_order gathers of W, G and H (:1033-1050)
//  - rq_writeback:        un-permute, dequantize, cast to the layer dtype, export buffers (:1850-1896)
// All of these are HBM-bound gathers / reductions.
#include <type_traits>

#include "rq_common.h"

namespace {

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = rq_nan_min(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = rq_nan_max(v, __shfl_xor(v, o, 64));
  return v;
}

// One wavefront per (row, group).
template <typename TW>
__global__ __launch_bounds__(256) void k_find_params(const TW* __restrict__ w, int R, int C,
                                                     int64_t ldw, int gs, float maxq, int sym, int clip_zero,
                                                     float* __restrict__ scale,
                                                     float* __restrict__ zero) {
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int grp = blockIdx.y;
  if (r >= R) return;
  const int c0 = grp * gs;
  const int c1 = min(C, c0 + gs);
  const TW* row = w + (int64_t)r * ldw;
  float mn = __builtin_inff(), mx = -__builtin_inff();
  // lane order c = c0 + lane, + 64, ... (the order decides which zero a min / max of +0 and -0
  // keeps); 8 loads in flight per lane
  int c = c0 + lane;
  for (; c + 7 * 64 < c1; c += 8 * 64) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = rq_load_elem(row + c + 64 * u);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      mn = rq_nan_min(mn, v[u]);
      mx = rq_nan_max(mx, v[u]);
    }
  }
  for (; c < c1; c += 64) {
    const float v = rq_load_elem(row + c);
    mn = rq_nan_min(mn, v);
    mx = rq_nan_max(mx, v);
  }
  mn = wave_min(mn);
  mx = wave_max(mx);
  if (lane == 0) {
    float s, z;
    rq_params_from_minmax(mn, mx, maxq, sym, &s, &z, clip_zero);
    scale[(int64_t)grp * R + r] = s;
    zero[(int64_t)grp * R + r] = z;
  }
}

// WeightQuantizer.find_params with mse=True (utils/quant_utils.py:408-448): min/max start,
// then a maxshrink*grid x maxshrink*grid shrink grid over (xmin, xmax); each candidate's row
// error sum |q - x|^norm is reduced in a fixed order and the first strict minimum wins
// (clip_zero = 0: the groupwise search of :354-386, from the group's own min / max).
//
// Bound by VALU issue: a candidate costs every element a divide, a round, a clamp and a power.
//  - Symmetric: s depends on (i, j) only through max(|xmin1|, xmax1), one of 2 * steps values, and
//    equal steps have equal errors, so 2 * steps candidates are evaluated instead of steps^2
//    (50 instead of 625 at the default grid).  Shrunk past zero (maxshrink > 1) the factors
//    change sign and |xmin1| no longer falls with i: there all steps^2 are evaluated.
//  - x / s with s shared by all elements: y = RN(1 / s), q0 = RN(x y), then one residual step
//    q0 + y (x - s q0) in two fused operations is the correctly rounded quotient (Markstein)
//    while nothing underflows; steps outside [2^-60, 2^60] take the IEEE divide.
//  - |q - x|^norm in 64-bit arithmetic (mse_pow), a quarter of powf's instructions.  Its last bit is
//    not powf's, so it settles only what it can: candidates whose error lies within the two sums'
//    rounding of the least are summed again with powf (and the IEEE divide), and those sums decide,
//    so the choice is the one that powf throughout makes.  The candidates in question are kept in
//    a list as they come (8 for each of a batch's places, a lane each); a wave whose list ran over
//    goes through its batches again.
//  - One wave per candidate batch: a lane holds 4 of 256 interleaved partial sums, and 8
//    candidates are reduced together by halving exchanges (10 shuffles instead of 48), with no
//    barrier.  Up to MSE_WIDE elements a wave owns one (row, group); wider rows share a
//    workgroup's 4 waves, which take every fourth batch.
// 1024 x 4096 fp32 against one 256-thread workgroup per (row, group), every candidate, the IEEE
// divide and powf: symmetric 16.3 -> 0.40 ms (128-column groups) and 10.7 -> 0.36 ms (per row),
// asymmetric 16.5 -> 4.1 and 10.5 -> 3.1 ms (of which the sums by powf 3 to 5 %, of symmetric rows 14 %).
constexpr int MSE_WIDE = 1024;          // above: one (row, group) per workgroup
constexpr int MSE_LDS_MAX = 16384;      // elements staged in LDS; wider groups are read in place
constexpr int MSE_B = 8;                // candidates per batch

struct MseLog {
  double inv, log2c;                    // 1 / c and log2(c) of an interval's centre c
};

// |d|^p for d >= 0 finite and p > 0, in 64 bits and rounded once: log2(d) = e + log2(c) +
// log2(m / c) with m / c - 1 within 0.0304 of 0 (a table of 16 centres c), 2^y by its
// fractional part.  Both polynomials were fitted for this kernel at Chebyshev nodes of their
// intervals (errors 2^-36 and 2^-34), so the result is within 0.5 + 2^-10 + p 2^-12 units of
// the last place (powf: 1).
__device__ __forceinline__ float mse_pow(float d, double p, const MseLog* tab) {
  const float m = __builtin_amdgcn_frexp_mantf(d);
  const int e = __builtin_amdgcn_frexp_expf(d);
  const MseLog t = tab[(__float_as_uint(m) >> 19) & 15];
  const double r = __builtin_fma((double)m, t.inv, -1.0);
  double a = 0x1.27c1ba5fe9d34p-2;
  a = __builtin_fma(a, r, -0x1.719d5484e3a26p-2);
  a = __builtin_fma(a, r, 0x1.ec70971caf89bp-2);
  a = __builtin_fma(a, r, -0x1.7154742aec3edp-1);
  a = __builtin_fma(a, r, 0x1.71547652bdc8bp+0);
  const double y = p * __builtin_fma(a, r, (double)e + t.log2c);
  const double n = __builtin_rint(y);
  const double f = y - n;
  double z = 1.531008147539287e-05;
  z = __builtin_fma(z, f, 0.00015469731991027595);
  z = __builtin_fma(z, f, 0.001333345055956001);
  z = __builtin_fma(z, f, 0.009618025602929684);
  z = __builtin_fma(z, f, 0.055504109412156666);
  z = __builtin_fma(z, f, 0.2402265121359518);
  z = __builtin_fma(z, f, 0.6931471805459303);
  z = __builtin_fma(z, f, 0.9999999999595488);
  const float v = (float)__builtin_amdgcn_ldexp(z, (int)n);
  return d == 0.0f ? 0.0f : v;
}

// No factor 1 - i / grid below zero.
__host__ __device__ constexpr bool mse_distinct(int grid, int steps) { return steps - 1 <= grid; }

// The step and zero of candidate c, and whether it is one of the grid's.  Distinct steps of a
// symmetric grid (DISTINCT, factors that fall from 1 and stay non-negative): c < steps is |xmin|
// shrunk by row c of the grid (where some column leaves xmax no larger), the others xmax shrunk by
// column c - steps.  Else candidate c is row c / steps, column c % steps.  (DISTINCT at run time:
// 2 % longer, 17 scalar registers more spilled.)
template <bool SYM, bool DISTINCT>
struct MseGrid {
  float xmin, xmax, maxq;
  int grid, steps, n;
  __device__ __forceinline__ float fac(int i) const { return (float)(1.0 - (double)i / (double)grid); }
  __device__ __forceinline__ float lo(int i) const { return fabsf(fac(i) * xmin); }
  __device__ __forceinline__ float hi(int j) const { return fac(j) * xmax; }
  __device__ __forceinline__ bool params(int c, float* s, float* z) const {
    if (DISTINCT) {
      const int k = c < steps ? c : c - steps;
      const float m = c < steps ? lo(k) : hi(k);
      // the other side's smallest value decides whether max() ever takes m
      const float other = c < steps ? rq_nan_min(hi(0), hi(steps - 1)) : lo(steps - 1);
      *s = rq_clamp_min(m, 1e-5f) / maxq;
      *z = 0.0f;
      // (both sides shrunk alike to one value: the row's)
      return c < n && !(other > m) && !(c >= steps && lo(k) == m);
    }
    const float xmin1 = fac(c / steps) * xmin, xmax1 = fac(c % steps) * xmax;
    if (SYM) {
      *s = rq_clamp_min(rq_nan_max(fabsf(xmin1), xmax1), 1e-5f) / maxq;
      *z = 0.0f;
      return c < n;
    }
    *s = (xmax1 - xmin1) / maxq;
    *z = __builtin_rintf(-xmin1 / *s);
    return c < n;
  }
  // place of candidate c in the search order (row by row), for equal errors
  __device__ int64_t first(int c) const {
    if (!DISTINCT) return c;
    const bool row = c < steps;
    const int k = row ? c : c - steps;
    const float m = row ? lo(k) : hi(k);
    int o = 0;
    while (o < steps - 1 && (row ? hi(o) : lo(o)) > m) ++o;
    return row ? (int64_t)k * steps + o : (int64_t)o * steps + k;
  }
};

// The element's code times the step (the rounded quotient t = x / s comes in).
template <bool SYM>
__device__ __forceinline__ float mse_quant(float t, float s, float z, float maxq) {
  t = __builtin_rintf(t);
  if (SYM) {
    t = (t < -(maxq + 1.0f)) ? -(maxq + 1.0f) : t;
    t = (t > maxq) ? maxq : t;
    return s * t;
  }
  t = t + z;
  t = (t < 0.0f) ? 0.0f : t;
  t = (t > maxq) ? maxq : t;
  return s * (t - z);
}

// One batch: the partial sums of MSE_B candidates over the lane's elements.
template <bool SYM, typename TX>
__device__ __forceinline__ void mse_batch(const TX* x, int n, int lane, const float* s, const float* z, const float* y,
                                          float maxq, double p, const MseLog* tab, float* part) {
  float acc[MSE_B][4];
#pragma unroll
  for (int k = 0; k < MSE_B; ++k)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[k][u] = 0.0f;
  for (int c0 = 0; c0 < n; c0 += 256) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (c0 + 64 * u >= n) break;                     // the same for the whole wave
      const int c = c0 + 64 * u + lane;
      const bool in = c < n;
      const float v = rq_load_elem(x + (in ? c : 0));
#pragma unroll
      for (int k = 0; k < MSE_B; ++k) {
        const float q0 = v * y[k];
        const float t = __builtin_fmaf(__builtin_fmaf(-s[k], q0, v), y[k], q0);
        const float e = mse_pow(fabsf(mse_quant<SYM>(t, s[k], z[k], maxq) - v), p, tab);
        acc[k][u] += in ? e : 0.0f;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < MSE_B; ++k) part[k] = (acc[k][0] + acc[k][2]) + (acc[k][1] + acc[k][3]);
}

// The same for one candidate with any step, norm and data: IEEE divide and powf.
template <bool SYM, typename TX>
__device__ __attribute__((noinline)) float mse_any(const TX* x, int n, int lane, float s, float z, float maxq,
                                                   float norm) {
  float sum[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    sum[u] = 0.0f;
    for (int c = 64 * u + lane; c < n; c += 256) {
      const float v = rq_load_elem(x + c);
      sum[u] += powf(fabsf(mse_quant<SYM>(v / s, s, z, maxq) - v), norm);
    }
  }
  return (sum[0] + sum[2]) + (sum[1] + sum[3]);
}

template <bool SYM, bool DISTINCT, typename TW, bool STAGED>
__global__ __launch_bounds__(256) void k_find_params_mse(const TW* __restrict__ w, int R, int C,
                                                         int64_t ldw, int gs, int ng, float maxq,
                                                         int clip_zero, float norm, int grid, int steps,
                                                         int per_wg, float* __restrict__ scale,
                                                         float* __restrict__ zero) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  __shared__ MseLog tab[16];
  __shared__ float best_e[4], best_e2[4];
  __shared__ int best_c[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid < 16) {
    const double c = 0.5 + (tid + 0.5) / 32.0;
    tab[tid].inv = 1.0 / c;
    tab[tid].log2c = log2(c);
  }
  __syncthreads();
  // per_wg 4: each wave its own (row, group); per_wg 1: the waves share one.  Grid: rows x groups.
  const bool shared = per_wg == 1;
  const int64_t item = shared ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wave;
  const bool live = item < (int64_t)R * ng;
  const int r = live ? (int)(item % R) : 0, grp = live ? (int)(item / R) : 0;
  const int c0 = grp * gs;
  const int n = live ? min(C, c0 + gs) - c0 : 0;
  const TW* row = w + (int64_t)r * ldw + c0;
  float* xw = xs + (shared ? 0 : wave * gs);
  if (STAGED) {
    for (int c = shared ? tid : lane; c < n; c += shared ? 256 : 64) xw[c] = rq_load_elem(row + c);
    __syncthreads();
  }
  auto elem = [&](int c) -> float { return STAGED ? xw[c] : rq_load_elem(row + c); };
  // min and max in the order of 256 interleaved lanes (it decides which of +0 and -0 is kept)
  float mn[4], mx[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    mn[u] = __builtin_inff();
    mx[u] = -__builtin_inff();
    for (int c = 64 * u + lane; c < n; c += 256) {
      mn[u] = rq_nan_min(mn[u], elem(c));
      mx[u] = rq_nan_max(mx[u], elem(c));
    }
  }
  float rmin = rq_nan_min(rq_nan_min(mn[0], mn[2]), rq_nan_min(mn[1], mn[3]));
  float rmax = rq_nan_max(rq_nan_max(mx[0], mx[2]), rq_nan_max(mx[1], mx[3]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    rmin = rq_nan_min(rmin, __shfl_down(rmin, o, 64));
    rmax = rq_nan_max(rmax, __shfl_down(rmax, o, 64));
  }
  rmin = __shfl(rmin, 0, 64);
  rmax = __shfl(rmax, 0, 64);
  MseGrid<SYM, DISTINCT> g;
  g.xmin = clip_zero ? rq_nan_min(rmin, 0.0f) : rmin;
  g.xmax = clip_zero ? rq_nan_max(rmax, 0.0f) : rmax;
  if (!SYM && g.xmin == 0.0f && g.xmax == 0.0f) {
    g.xmin = -1.0f;
    g.xmax = 1.0f;
  }
  g.maxq = maxq;
  g.grid = grid;
  g.steps = steps;
  g.n = !live ? 0 : DISTINCT ? 2 * steps : steps * steps;
  // one step only, the start's (its lower bound), or no error at all: the first candidate wins
  if (DISTINCT && rq_nan_max(fabsf(g.xmin), g.xmax) <= 1e-5f) g.n = 0;
  if (!SYM && rmin == 0.0f && rmax == 0.0f) g.n = min(g.n, 1);
  const double p = (double)norm;
  const bool fast = norm > 0.0f && norm < 64.0f;
  // the lane's own candidate among the batch's: bit 5, 4, 3 of the lane
  const int mine = ((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1);
  // The least error and its candidate, and the next least: of the 8 lanes that share `mine`, then
  // of all.
  float be = __builtin_inff(), be2 = __builtin_inff();
  int bc = -1;
  auto take = [&](float e, int c) {
    const bool less = e < be || (e == be && bc >= 0 && g.first(c) < g.first(bc));
    const float other = less ? be : e;
    be2 = other < be2 ? other : be2;
    be = less ? e : be;
    bc = less ? c : bc;
  };
  // Errors within near(least) of each other are in question: n terms that differ by 2 units of
  // the last place at most (a unit is 2^-23; and 2 subnormal ones), in sums of n / 256 + 9
  // roundings each.  near - 1 is over twice the sums' largest relative difference.
  const float slack = (float)((n + 255) / 256 + 16) * 0x1p-21f, least_e = (float)n * 0x1p-147f;
  auto near = [&](float e) { return e + e * slack + least_e; };
  // the list: lane q of the 8 holds entry q
  float list_e = 0.0f;
  int list_c = 0, listed = 0;
  auto all_lanes = [&](float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
  };
  auto merge = [&](float oe, int oc, float oe2) {
    if (oc >= 0) take(oe, oc);
    be2 = oe2 < be2 ? oe2 : be2;
  };
  auto merge_waves = [&]() {
    if (!shared) return;
    if (lane == 0) {
      best_e[wave] = be;
      best_e2[wave] = be2;
      best_c[wave] = bc;
    }
    __syncthreads();
    be = best_e[0];
    be2 = best_e2[0];
    bc = best_c[0];
    for (int k = 1; k < 4; ++k) merge(best_e[k], best_c[k], best_e2[k]);
    __syncthreads();
  };
  // a candidate by powf: the lane's part of the sum
  auto any = [&](float sk, float zk) {
    return STAGED ? mse_any<SYM>(xw, n, lane, sk, zk, maxq, norm) : mse_any<SYM>(row, n, lane, sk, zk, maxq, norm);
  };
  // the candidates c of the lanes in `todo`
  auto evaluate = [&](uint64_t todo, int c) {
    for (; todo; todo &= todo - 1) {
      const int l = __builtin_ctzll(todo), cl = __builtin_amdgcn_readlane(c, l);
      if (be == 0.0f && bc >= 0 && g.first(cl) > g.first(bc)) continue;      // not less than nothing
      float sk, zk;
      g.params(cl, &sk, &zk);
      take(all_lanes(any(sk, zk)), cl);
    }
  };
  bool settled = false;
  // Pass 0: every candidate, by mse_pow.  Pass 1 (a list that ran over): those in question, by powf.
  float limit = 0.0f;
  for (int pass = 0; pass < 2; ++pass) {
    for (int b = shared ? wave : 0; b * MSE_B < g.n; b += shared ? 4 : 1) {
      // lane k < 8 works out candidate k's step; every lane then reads all eight
      float cs, cz;
      const bool ok = g.params(b * MSE_B + (lane & (MSE_B - 1)), &cs, &cz);
      const float cy = 1.0f / cs;
      // steps for which the residual divide is exact, and finite data (an infinity or NaN in the
      // row makes every step one)
      const bool good = fast && cs >= 0x1p-60f && cs <= 0x1p60f;
      float s[MSE_B], z[MSE_B], y[MSE_B], part[MSE_B];
#pragma unroll
      for (int k = 0; k < MSE_B; ++k) {
        s[k] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(cs), k));
        z[k] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(cz), k));
        y[k] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(cy), k));
      }
      const uint64_t valid = __ballot(ok) & 255, exact = __ballot(good || !ok) & 255;
      if (!valid) continue;
      if (exact == 255) {
        if (STAGED) mse_batch<SYM>(xw, n, lane, s, z, y, maxq, p, tab, part);
        else mse_batch<SYM>(row, n, lane, s, z, y, maxq, p, tab, part);
      } else {
        for (int k = 0; k < MSE_B; ++k) {
          const float sk = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(cs), k));
          const float zk = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(cz), k));
          const float v = any(sk, zk);
#pragma unroll
          for (int j = 0; j < MSE_B; ++j)
            if (j == k) part[j] = v;
        }
      }
      // the tree of 64 partial sums (l + (l + 32), + 16, ...), halving the candidates a lane keeps
      // for the first three levels; each lane ends with the sum of candidate `mine`
      float h4[4], h2[2];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool up = lane & 32;
        const float keep = up ? part[k + 4] : part[k], send = up ? part[k] : part[k + 4];
        h4[k] = keep + __shfl_xor(send, 32, 64);
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const bool up = lane & 16;
        const float keep = up ? h4[k + 2] : h4[k], send = up ? h4[k] : h4[k + 2];
        h2[k] = keep + __shfl_xor(send, 16, 64);
      }
      const bool up = lane & 8;
      float err = (up ? h2[1] : h2[0]) + __shfl_xor(up ? h2[0] : h2[1], 8, 64);
      err += __shfl_xor(err, 4, 64);
      err += __shfl_xor(err, 2, 64);
      err += __shfl_xor(err, 1, 64);
      const bool there = (valid >> mine) & 1;
      const int c = b * MSE_B + mine;
      if (pass == 0) {
        if (there && err <= near(be)) {
          if (be > near(err)) listed = 0;
          if ((lane & 7) == listed) {
            list_e = err;
            list_c = c;
          }
          ++listed;
        }
        if (there) take(err, c);
      } else {
        evaluate(__ballot(there && err <= limit && (lane & 7) == 0), c);
      }
    }
    if (pass == 1) break;
#pragma unroll
    for (int o = 32; o >= 8; o >>= 1) {
      const float oe = __shfl_xor(be, o, 64), oe2 = __shfl_xor(be2, o, 64);
      const int oc = __shfl_xor(bc, o, 64);
      merge(oe, oc, oe2);
    }
    merge_waves();
    limit = near(be);
    settled = !fast || be2 > limit;                     // (the same in all waves of a (row, group))
    if (settled) break;
    be = be2 = __builtin_inff();
    bc = -1;
    if (__ballot(listed > 8)) continue;
    evaluate(__ballot((lane & 7) < listed && list_e <= limit), list_c);
    break;
  }
  if (!settled) merge_waves();
  if (live && lane == 0 && (!shared || wave == 0)) {
    float bs, bz;
    if (bc >= 0) g.params(bc, &bs, &bz);
    else rq_params_from_minmax(rmin, rmax, maxq, SYM, &bs, &bz, clip_zero);
    scale[(int64_t)grp * R + r] = bs;
    zero[(int64_t)grp * R + r] = bz;
  }
}

template <typename TW>
__global__ __launch_bounds__(256) void k_gather_w(const TW* __restrict__ w, int64_t ldw,
                                                  const float* __restrict__ Hg, int R_s, int C,
                                                  const int64_t* __restrict__ perm,
                                                  float* __restrict__ out, int64_t ldo) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= C) return;
  const int64_t p = perm ? perm[j] : j;
  const bool dead = Hg[p * C + p] == 0.0f;
  for (int r = blockIdx.y; r < R_s; r += gridDim.y)
    out[(int64_t)r * ldo + j] = dead ? 0.0f : rq_load_elem(w + (int64_t)r * ldw + p);
}

__global__ __launch_bounds__(256) void k_gather_g(const float* __restrict__ g, int64_t ldg, int R_s,
                                                  int C, const int64_t* __restrict__ perm,
                                                  float* __restrict__ out, int64_t ldo) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= C) return;
  const int64_t p = perm ? perm[j] : j;
  for (int r = blockIdx.y; r < R_s; r += gridDim.y) out[(int64_t)r * ldo + j] = g[(int64_t)r * ldg + p];
}

// Row-staged gathers.  A workgroup copies `nr` whole source rows into LDS (16-byte loads when
// the rows allow, 8 in flight per thread), then writes the output rows in order, column j
// taking LDS element perm[j]: every source byte is read from HBM once and the writes are
// coalesced.  The column kernels above (the fallback for rows too wide for LDS) read one
// element per thread from anywhere in its row, fetching each row's cache lines once per
// 256-column workgroup.  Row stride in LDS: C elements rounded up to 16 bytes.
template <typename TS>
__host__ __device__ constexpr int padded_cols(int C) {
  return (int)(((int64_t)C * (int64_t)sizeof(TS) + 15) / 16 * 16 / (int64_t)sizeof(TS));
}

template <int NT, typename TS>
__device__ __forceinline__ void stage_rows(const TS* __restrict__ src, int64_t lds, int r0, int nr, int C,
                                           bool vec, uint8_t* smem) {
  const int tid = threadIdx.x;
  const int cpad = padded_cols<TS>(C);
  if (vec) {
    const int n16 = (int)((int64_t)C * sizeof(TS) / 16);
    const int rb = cpad * (int)sizeof(TS);
    const int tot = nr * n16;
    for (int q0 = tid; q0 < tot; q0 += NT * 8) {
      uint4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int q = q0 + NT * u;
        if (q < tot)
          v[u] = reinterpret_cast<const uint4*>(src + (int64_t)(r0 + q / n16) * lds)[q % n16];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int q = q0 + NT * u;
        if (q < tot) reinterpret_cast<uint4*>(smem + (int64_t)(q / n16) * rb)[q % n16] = v[u];
      }
    }
  } else {
    TS* buf = reinterpret_cast<TS*>(smem);
    for (int rr = 0; rr < nr; ++rr)
      for (int q = tid; q < C; q += NT) buf[(int64_t)rr * cpad + q] = src[(int64_t)(r0 + rr) * lds + q];
  }
}

// Source column of each output column for the row-staged gathers: idx_w[j] = perm[j], or -1
// for a dead column (H_g[perm[j], perm[j]] == 0: W's column is zeroed), idx_g[j] = perm[j].
// Written once per subgroup into H_sub's first 2 C words, which k_gather_h_rows overwrites
// afterwards on the same stream; the row gathers then read one coalesced index per column
// instead of perm[j] and a diagonal element of H_g each.
__global__ __launch_bounds__(256) void k_gather_index(const float* __restrict__ Hg, int C,
                                                      const int64_t* __restrict__ perm, int32_t* __restrict__ idx_w,
                                                      int32_t* __restrict__ idx_g) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= C) return;
  const int64_t p = perm ? perm[j] : j;
  idx_w[j] = (Hg[p * C + p] == 0.0f) ? -1 : (int32_t)p;
  idx_g[j] = (int32_t)p;
}

// out[r, j] = src[r, idx[j]] (0 where idx[j] < 0) for rows r0 .. r0 + nr - 1: k_gather_w /
// k_gather_g by rows.  NT threads (1024 for rows that leave room for only one or two
// workgroups per CU); GU columns' index loads in flight per thread.
constexpr int GU = 8;
template <int NT, typename TS>
__global__ __launch_bounds__(NT) void k_gather_rows(const TS* __restrict__ src, int64_t lds, int rows, int C,
                                                    int rpw, bool vec, const int32_t* __restrict__ idx,
                                                    float* __restrict__ out, int64_t ldo) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int r0 = blockIdx.x * rpw;
  const int nr = min(rpw, rows - r0);
  stage_rows<NT>(src, lds, r0, nr, C, vec, smem);
  __syncthreads();
  const TS* buf = reinterpret_cast<const TS*>(smem);
  const int cpad = padded_cols<TS>(C);
  for (int j0 = threadIdx.x; j0 < C; j0 += NT * GU) {
    int p[GU];
#pragma unroll
    for (int u = 0; u < GU; ++u) {
      const int j = j0 + NT * u;
      p[u] = (j < C) ? idx[j] : 0;
    }
    for (int rr = 0; rr < nr; ++rr)
#pragma unroll
      for (int u = 0; u < GU; ++u) {
        const int j = j0 + NT * u;
        if (j < C)
          out[(int64_t)(r0 + rr) * ldo + j] = (p[u] < 0) ? 0.0f : rq_load_elem(buf + (int64_t)rr * cpad + p[u]);
      }
  }
}

__global__ __launch_bounds__(256) void k_gather_h(const float* __restrict__ Hg, int C,
                                                  const int64_t* __restrict__ perm,
                                                  float* __restrict__ out) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= C) return;
  const int64_t pj = perm ? perm[j] : j;
  for (int i = blockIdx.y; i < C; i += gridDim.y) {
    const int64_t pi = perm ? perm[i] : i;
    float v = Hg[pi * C + pj];
    if (i == j && v == 0.0f) v = 1.0f;            // H_sub[dead, dead] = 1
    out[(int64_t)i * C + j] = v;
  }
}

// P H P by rows: workgroup i stages source row perm[i] in LDS with 16-byte loads (the whole
// row, C floats), then writes output row i coalesced, column j taking LDS word perm[j].
// Each source row is read from HBM once; the column-gather kernel above re-read every source
// row's cache lines once per 256-column workgroup.  Dynamic LDS: C * 4 bytes (112 KB at
// C = 28672, one workgroup per CU), so there both loops keep GR_U loads per thread in flight;
// small rows run unrolled once with 256 threads and several workgroups per CU instead.
template <int GR_THREADS, int GR_U>
__global__ __launch_bounds__(GR_THREADS) void k_gather_h_rows(const float* __restrict__ Hg, int C,
                                                              const int64_t* __restrict__ perm,
                                                              float* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) float row[];
  const int i = blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t pi = perm ? perm[i] : i;
  const float* src = Hg + pi * C;
  if ((C & 3) == 0) {
    const float4* s4 = reinterpret_cast<const float4*>(src);
    const int n4 = C / 4;
    for (int q0 = tid; q0 < n4; q0 += GR_THREADS * GR_U) {
      float4 v[GR_U];
#pragma unroll
      for (int u = 0; u < GR_U; ++u) {
        const int q = q0 + u * GR_THREADS;
        if (q < n4) v[u] = s4[q];
      }
#pragma unroll
      for (int u = 0; u < GR_U; ++u) {
        const int q = q0 + u * GR_THREADS;
        if (q < n4) reinterpret_cast<float4*>(row)[q] = v[u];
      }
    }
  } else {
    for (int q = tid; q < C; q += GR_THREADS) row[q] = src[q];
  }
  __syncthreads();
  float* dst = out + (int64_t)i * C;
  for (int j0 = tid; j0 < C; j0 += GR_THREADS * GR_U) {
    int pj[GR_U];
#pragma unroll
    for (int u = 0; u < GR_U; ++u) {
      const int j = j0 + u * GR_THREADS;
      pj[u] = (j < C) ? (perm ? (int)perm[j] : j) : 0;
    }
#pragma unroll
    for (int u = 0; u < GR_U; ++u) {
      const int j = j0 + u * GR_THREADS;
      if (j < C) {
        float v = row[pj[u]];
        if (j == i && v == 0.0f) v = 1.0f;        // H_sub[dead, dead] = 1
        dst[j] = v;
      }
    }
  }
}

template <typename TQ>
__global__ __launch_bounds__(256) void k_writeback(const int16_t* __restrict__ codes, int R, int C,
                                                   const int64_t* __restrict__ invperm, int qmode,
                                                   const float* __restrict__ scale,
                                                   const int32_t* __restrict__ col_group,
                                                   const float* __restrict__ dyn_scale, int bs,
                                                   TQ* __restrict__ q_out, int64_t ldq,
                                                   float* __restrict__ w_int_out,
                                                   float* __restrict__ scale_out,
                                                   int* __restrict__ nan_flag) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= C) return;
  const int64_t j = invperm ? invperm[c] : c;
  int nan_seen = 0;
  for (int r = blockIdx.y; r < R; r += gridDim.y) {
    const int16_t ci = codes[(int64_t)r * C + j];
    const float code = (ci == RQ_CODE_NAN) ? __builtin_nanf("") : (float)ci;   // NaN weight
    float s;
    if (qmode == RQ_QMODE_CHANNEL) s = scale[r];
    else if (qmode == RQ_QMODE_STATIC) s = scale[(int64_t)col_group[j] * R + r];
    else s = dyn_scale[(j / bs) * (int64_t)R + r];
    float qf = s * code;
    // Keep fl32(s * code) as its own rounding step: without the barrier the compiler folds
    // the multiply and the fp16 conversion into v_fma_mixlo_f16 (a single rounding), which
    // differs from torch's (scale * q).to(float16) on exact fp16 midpoints.
    asm volatile("" : "+v"(qf));
    const TQ q = rq_cast<TQ>(qf);
    q_out[(int64_t)r * ldq + c] = q;
    const float qback = (float)q;
    nan_seen |= (qback != qback);
    if (w_int_out) w_int_out[(int64_t)r * C + c] = code;
    if (scale_out) scale_out[(int64_t)r * C + c] = s;
  }
  if (nan_seen && nan_flag) atomicOr(nan_flag, 1);
}

// k_writeback by rows: the workgroup's rows of codes staged in LDS (as k_gather_rows), then
// each output row written in order, column c taking LDS element invperm[c]; the same
// arithmetic as k_writeback.
template <int NT, typename TQ>
__global__ __launch_bounds__(NT) void k_writeback_rows(const int16_t* __restrict__ codes, int R, int C, int rpw,
                                                        bool vec, const int64_t* __restrict__ invperm, int qmode,
                                                        const float* __restrict__ scale,
                                                        const int32_t* __restrict__ col_group,
                                                        const float* __restrict__ dyn_scale, int bs,
                                                        TQ* __restrict__ q_out, int64_t ldq,
                                                        float* __restrict__ w_int_out,
                                                        float* __restrict__ scale_out,
                                                        int* __restrict__ nan_flag) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int r0 = blockIdx.x * rpw;
  const int nr = min(rpw, R - r0);
  stage_rows<NT>(codes, C, r0, nr, C, vec, smem);
  __syncthreads();
  const int16_t* buf = reinterpret_cast<const int16_t*>(smem);
  const int cpad = padded_cols<int16_t>(C);
  int nan_seen = 0;
  constexpr int WU = 4;   // columns whose index loads are in flight per thread
  for (int c0 = threadIdx.x; c0 < C; c0 += NT * WU) {
    int64_t jj[WU], gb[WU];
#pragma unroll
    for (int u = 0; u < WU; ++u) {
      const int c = c0 + NT * u;
      jj[u] = (c < C) ? (invperm ? invperm[c] : c) : 0;
    }
#pragma unroll
    for (int u = 0; u < WU; ++u)
      gb[u] = (qmode == RQ_QMODE_STATIC)  ? (int64_t)col_group[jj[u]] * R
              : (qmode == RQ_QMODE_DYNAMIC) ? (jj[u] / bs) * (int64_t)R
                                            : 0;
    for (int rr = 0; rr < nr; ++rr) {
#pragma unroll
      for (int u = 0; u < WU; ++u) {
        const int c = c0 + NT * u;
        if (c >= C) continue;
        const int64_t j = jj[u], gbase = gb[u];
        const int r = r0 + rr;
        const int16_t ci = buf[(int64_t)rr * cpad + j];
        const float code = (ci == RQ_CODE_NAN) ? __builtin_nanf("") : (float)ci;   // NaN weight
        float s;
        if (qmode == RQ_QMODE_CHANNEL) s = scale[r];
        else if (qmode == RQ_QMODE_STATIC) s = scale[gbase + r];
        else s = dyn_scale[gbase + r];
        float qf = s * code;
        asm volatile("" : "+v"(qf));   // fl32(s * code), then the cast: two roundings (k_writeback)
        const TQ q = rq_cast<TQ>(qf);
        q_out[(int64_t)r * ldq + c] = q;
        const float qback = (float)q;
        nan_seen |= (qback != qback);
        if (w_int_out) w_int_out[(int64_t)r * C + c] = code;
        if (scale_out) scale_out[(int64_t)r * C + c] = s;
      }
    }
  }
  if (nan_seen && nan_flag) atomicOr(nan_flag, 1);
}

inline int rows_grid(int rows) { return rows < 1024 ? rows : 1024; }

// Rows per workgroup and LDS bytes of a row-staged launch over `rows` rows of C elements of
// `esize` bytes: enough workgroups to keep ~1024 in the grid, at most 4 rows and 64 KB; 0 when
// one row does not fit the LDS a workgroup may have (then the column kernels run).
template <typename K>
inline size_t rows_launch(K kernel, int rows, int C, int esize, int* rpw) {
  const size_t rb = (size_t)(((int64_t)C * esize + 15) / 16 * 16);
  int n = rows / 1024;
  n = n < 1 ? 1 : (n > 4 ? 4 : n);
  while (n > 1 && (size_t)n * rb > 64 * 1024) --n;
  const size_t bytes = (size_t)n * rb;
  if (bytes > 64 * 1024 &&
      (bytes > 160 * 1024 ||
       hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess))
    return 0;
  *rpw = n;
  return bytes;
}

// 16-byte row loads: the row length and stride are whole 16-byte units and the base is aligned.
inline bool rows_vec(const void* p, int64_t ld, int C, int esize) {
  return ((int64_t)C * esize) % 16 == 0 && (ld * esize) % 16 == 0 && ((uintptr_t)p & 15) == 0;
}

// 256 threads per workgroup while a row is at most 32 KB, else 1024 (LDS then holds one or
// two workgroups per CU).
inline bool rows_wide(int C, int esize) { return (int64_t)C * esize > 32 * 1024; }

template <typename TS>
inline bool launch_gather_rows(const TS* src, int64_t lds, int rows, int C, const int32_t* idx, float* out,
                               int64_t ldo, hipStream_t s) {
  int rpw = 1;
  const bool vec = rows_vec(src, lds, C, (int)sizeof(TS));
  if (rows_wide(C, (int)sizeof(TS))) {
    const size_t bytes = rows_launch(k_gather_rows<1024, TS>, rows, C, (int)sizeof(TS), &rpw);
    if (!bytes) return false;
    hipLaunchKernelGGL((k_gather_rows<1024, TS>), dim3((rows + rpw - 1) / rpw), dim3(1024), bytes, s, src, lds,
                       rows, C, rpw, vec, idx, out, ldo);
  } else {
    const size_t bytes = rows_launch(k_gather_rows<256, TS>, rows, C, (int)sizeof(TS), &rpw);
    if (!bytes) return false;
    hipLaunchKernelGGL((k_gather_rows<256, TS>), dim3((rows + rpw - 1) / rpw), dim3(256), bytes, s, src, lds,
                       rows, C, rpw, vec, idx, out, ldo);
  }
  return true;
}

// Groups up to MSE_WIDE elements: a wave each, four per workgroup; wider ones a workgroup each;
// staged in LDS up to MSE_LDS_MAX elements (64 KB).
template <typename TW>
int launch_find_params_mse(const TW* w, int R, int C, int64_t ldw, int gs, int ng, int maxq, int sym, int clip_zero,
                           float norm, int grid, int steps, float* scale, float* zero, hipStream_t s) {
  const int width = gs < C ? gs : C;
  const int per_wg = width <= MSE_WIDE ? 4 : 1;
  const int64_t items = (int64_t)R * ng, wgs = (items + per_wg - 1) / per_wg;
  const bool distinct = sym && mse_distinct(grid, steps);
  // candidates are counted in 32 bits (46340^2 < 2^31)
  if (wgs > 0x7fffffff || steps > (distinct ? 1 << 29 : 46340)) return RQ_EINVAL;
  const bool staged = width <= MSE_LDS_MAX;
  const size_t lds = staged ? (size_t)per_wg * width * sizeof(float) : 0;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(256), lds, s, w, R, C, ldw, width, ng, (float)maxq, clip_zero,
                       norm, grid, steps, per_wg, scale, zero);
  };
  if (distinct && staged) go(k_find_params_mse<true, true, TW, true>);
  else if (distinct) go(k_find_params_mse<true, true, TW, false>);
  else if (sym && staged) go(k_find_params_mse<true, false, TW, true>);
  else if (sym) go(k_find_params_mse<true, false, TW, false>);
  else if (staged) go(k_find_params_mse<false, false, TW, true>);
  else go(k_find_params_mse<false, false, TW, false>);
  RQ_CHECK_LAUNCH();
  return RQ_OK;
}

}  // namespace

extern "C" int rq_find_params(const void* w, int w_dtype, int R, int C, int64_t ldw, int group_size,
                              int maxq, int sym, int clip_zero, float* scale, float* zero, void* stream) {
  if (!w || !scale || !zero || R <= 0 || C <= 0 || ldw < C || maxq <= 0) return RQ_EINVAL;
  const int gs = group_size > 0 ? group_size : C;
  const int ng = (C + gs - 1) / gs;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  dim3 grid((R + 3) / 4, ng), block(256);
  if (w_dtype == RQ_F16)
    hipLaunchKernelGGL(k_find_params<__half>, grid, block, 0, s, (const __half*)w, R, C, ldw, gs,
                       (float)maxq, sym, clip_zero, scale, zero);
  else if (w_dtype == RQ_BF16)
    hipLaunchKernelGGL(k_find_params<__hip_bfloat16>, grid, block, 0, s, (const __hip_bfloat16*)w, R,
                       C, ldw, gs, (float)maxq, sym, clip_zero, scale, zero);
  else if (w_dtype == RQ_F32)
    hipLaunchKernelGGL(k_find_params<float>, grid, block, 0, s, (const float*)w, R, C, ldw, gs,
                       (float)maxq, sym, clip_zero, scale, zero);
  else
    return RQ_EINVAL;
  RQ_CHECK_LAUNCH();
  return RQ_OK;
}

extern "C" int rq_find_params_mse(const void* w, int w_dtype, int R, int C, int64_t ldw,
                                  int group_size, int maxq, int sym, int clip_zero, double norm, int grid,
                                  double maxshrink, float* scale, float* zero, void* stream) {
  if (!w || !scale || !zero || R <= 0 || C <= 0 || ldw < C || maxq <= 0 || grid <= 0) return RQ_EINVAL;
  const int gs = group_size > 0 ? group_size : C;
  const int ng = (C + gs - 1) / gs;
  const int steps = (int)(maxshrink * grid);   // int(self.maxshrink * self.grid)
  if (steps <= 0) return RQ_EINVAL;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (w_dtype == RQ_F16)
    return launch_find_params_mse((const __half*)w, R, C, ldw, gs, ng, maxq, sym, clip_zero, (float)norm, grid, steps,
                                  scale, zero, s);
  if (w_dtype == RQ_BF16)
    return launch_find_params_mse((const __hip_bfloat16*)w, R, C, ldw, gs, ng, maxq, sym, clip_zero, (float)norm,
                                  grid, steps, scale, zero, s);
  if (w_dtype == RQ_F32)
    return launch_find_params_mse((const float*)w, R, C, ldw, gs, ng, maxq, sym, clip_zero, (float)norm, grid, steps,
                                  scale, zero, s);
  return RQ_EINVAL;
}

extern "C" int rq_prepare_subgroup(const void* w, int w_dtype, int64_t ldw, const float* grad,
                                   int64_t ldg, const float* H_g, int R_s, int C,
                                   const int64_t* perm, float* W_sub, int64_t ld_wsub, float* G_sub,
                                   int64_t ld_gsub, float* H_sub, void* stream) {
  if (!w || !H_g || !W_sub || !H_sub || R_s <= 0 || C <= 0 || ldw < C || ld_wsub < C) return RQ_EINVAL;
  if (grad && (!G_sub || ldg < C || ld_gsub < C)) return RQ_EINVAL;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  dim3 gw((C + 255) / 256, rows_grid(R_s)), block(256);
  // the source-column indices of the row gathers, in H_sub's first 2 C words (C >= 2), which
  // the H gather below overwrites after the W / G gathers have read them (same stream)
  int32_t* idx_w = reinterpret_cast<int32_t*>(H_sub);
  int32_t* idx_g = idx_w + C;
  const bool by_rows = C >= 2 && (uintptr_t)H_sub % 4 == 0;
  if (by_rows) {
    hipLaunchKernelGGL(k_gather_index, dim3((C + 255) / 256), block, 0, s, H_g, C, perm, idx_w, idx_g);
    RQ_CHECK_LAUNCH();
  }
  if (w_dtype == RQ_F16) {
    if (!by_rows || !launch_gather_rows((const __half*)w, ldw, R_s, C, idx_w, W_sub, ld_wsub, s))
      hipLaunchKernelGGL(k_gather_w<__half>, gw, block, 0, s, (const __half*)w, ldw, H_g, R_s, C, perm,
                         W_sub, ld_wsub);
  } else if (w_dtype == RQ_BF16) {
    if (!by_rows || !launch_gather_rows((const __hip_bfloat16*)w, ldw, R_s, C, idx_w, W_sub, ld_wsub, s))
      hipLaunchKernelGGL(k_gather_w<__hip_bfloat16>, gw, block, 0, s, (const __hip_bfloat16*)w, ldw, H_g,
                         R_s, C, perm, W_sub, ld_wsub);
  } else if (w_dtype == RQ_F32) {
    if (!by_rows || !launch_gather_rows((const float*)w, ldw, R_s, C, idx_w, W_sub, ld_wsub, s))
      hipLaunchKernelGGL(k_gather_w<float>, gw, block, 0, s, (const float*)w, ldw, H_g, R_s, C, perm,
                         W_sub, ld_wsub);
  } else {
    return RQ_EINVAL;
  }
  RQ_CHECK_LAUNCH();
  if (grad) {
    if (!by_rows || !launch_gather_rows(grad, ldg, R_s, C, idx_g, G_sub, ld_gsub, s))
      hipLaunchKernelGGL(k_gather_g, gw, block, 0, s, grad, ldg, R_s, C, perm, G_sub, ld_gsub);
    RQ_CHECK_LAUNCH();
  }
  const size_t row_bytes = (size_t)C * sizeof(float);
  if (row_bytes <= 64 * 1024 ||
      (row_bytes <= 160 * 1024 &&
       hipFuncSetAttribute((const void*)k_gather_h_rows<512, 8>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)row_bytes) == hipSuccess)) {
    if (C >= 8192)
      hipLaunchKernelGGL((k_gather_h_rows<512, 8>), dim3(C), dim3(512), row_bytes, s, H_g, C, perm, H_sub);
    else
      hipLaunchKernelGGL((k_gather_h_rows<256, 1>), dim3(C), dim3(256), row_bytes, s, H_g, C, perm, H_sub);
  } else {
    hipLaunchKernelGGL(k_gather_h, dim3((C + 255) / 256, rows_grid(C)), block, 0, s, H_g, C, perm, H_sub);
  }
  RQ_CHECK_LAUNCH();
  return RQ_OK;
}

extern "C" int rq_writeback(const int16_t* codes, int R, int C, const int64_t* invperm, int qmode,
                            const float* scale, const int32_t* col_group, const float* dyn_scale,
                            int blocksize, void* q_out, int q_dtype, int64_t ldq, float* w_int_out,
                            float* scale_out, int* nan_flag, void* stream) {
  if (!codes || !q_out || R <= 0 || C <= 0 || ldq < C) return RQ_EINVAL;
  if (qmode == RQ_QMODE_CHANNEL && !scale) return RQ_EINVAL;
  if (qmode == RQ_QMODE_STATIC && (!scale || !col_group)) return RQ_EINVAL;
  if (qmode == RQ_QMODE_DYNAMIC && (!dyn_scale || blocksize <= 0)) return RQ_EINVAL;
  if (qmode < 0 || qmode > 2) return RQ_EINVAL;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  dim3 grid((C + 255) / 256, rows_grid(R)), block(256);
  // by rows when a row of codes fits the LDS of a workgroup, else the column kernel
  auto run = [&](auto* q) -> int {
    typedef typename std::remove_pointer<decltype(q)>::type TQ;
    int rpw = 1;
    const bool vec = rows_vec(codes, C, C, (int)sizeof(int16_t));
    const bool wide = rows_wide(C, (int)sizeof(int16_t));
    const size_t bytes = wide ? rows_launch(k_writeback_rows<1024, TQ>, R, C, (int)sizeof(int16_t), &rpw)
                              : rows_launch(k_writeback_rows<256, TQ>, R, C, (int)sizeof(int16_t), &rpw);
    if (bytes && wide)
      hipLaunchKernelGGL((k_writeback_rows<1024, TQ>), dim3((R + rpw - 1) / rpw), dim3(1024), bytes, s, codes, R,
                         C, rpw, vec, invperm, qmode, scale, col_group, dyn_scale, blocksize, q, ldq, w_int_out,
                         scale_out, nan_flag);
    else if (bytes)
      hipLaunchKernelGGL((k_writeback_rows<256, TQ>), dim3((R + rpw - 1) / rpw), block, bytes, s, codes, R, C,
                         rpw, vec, invperm, qmode, scale, col_group, dyn_scale, blocksize, q, ldq, w_int_out,
                         scale_out, nan_flag);
    else
      hipLaunchKernelGGL(k_writeback<TQ>, grid, block, 0, s, codes, R, C, invperm, qmode, scale, col_group,
                         dyn_scale, blocksize, q, ldq, w_int_out, scale_out, nan_flag);
    return RQ_OK;
  };
  if (q_dtype == RQ_F16)
    run((__half*)q_out);
  else if (q_dtype == RQ_BF16)
    run((__hip_bfloat16*)q_out);
  else if (q_dtype == RQ_F32)
    run((float*)q_out);
  else
    return RQ_EINVAL;
  RQ_CHECK_LAUNCH();
  return RQ_OK;
}
