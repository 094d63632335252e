// Kernels of the per-site log sums shared by the linear_c.c twins: the
// util vector of ten_log_like3_c / ten_*_logdot_c / mat_* and its
// sequential log sum.  Internal linkage, so that every translation unit that
// launches them holds its own copy of the same code.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "pp_crmath.h"
#include "pp_exact_sum.h"

namespace pp {

// per-site util of ten_log_like3_c (statd != null) or ten_*_logdot_c;
// sites [first, first+n_used), optional mask.  One lane per site, as the sum
// over (rate, state) is sequential; S known (4, 20) keeps a rate's loads in
// flight together, S = 0 takes any number of states.
template <int S>
static __global__ void util_kernel(double *util, const double *statd, const double *x, const double *y,
                                   const double *z, const uint16_t *mask, int first, int n_used, int R,
                                   int N, int any_S) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_used) return;
  const int site = first + t;
  double u = 0.0;
  if (!mask || mask[site]) {
    const int states = S ? S : any_S;
    for (int r = 0; r < R; r++) {
      const long o = ((long)r * N + site) * states;
      if constexpr (S > 0) {
        double a[S], b[S], c[S];
#pragma unroll
        for (int s = 0; s < S; s++) {
          a[s] = x[o + s];
          b[s] = y[o + s];
          if (statd) c[s] = z[o + s];
        }
#pragma unroll
        for (int s = 0; s < S; s++) u = statd ? u + ((statd[s] * a[s]) * b[s]) * c[s] : u + a[s] * b[s];
      } else {
        for (int s = 0; s < states; s++) {
          if (statd) u = u + ((statd[s] * x[o + s]) * y[o + s]) * z[o + s];
          else u = u + x[o + s] * y[o + s];
        }
      }
    }
  }
  util[t] = u;
}

// sequential site-order log sum (linear_c.c:416-421 / 527-536) of correctly
// rounded logs (pp_crmath.h), as the stubs' libm returns them; the mat_*
// stubs (linear_c.c:170-340) have no n log R term (rate_term = 0).  With
// exponents xe, ye (and ze): the GLV functions' value, plus log 2 times their
// site-order float sums (total_twoexp / masked_total_twoexp /
// bounded_total_twoexp, gstar_support.ml:47-70; sums of integers, exact in any
// order).
//
// One workgroup: its lanes take the logs of 4,096 sites at a time into LDS and
// the first wave adds them in site order (wave_sequential_sum, going on from
// the sum so far).  With one lane for both, 1,601 sites took 680 us, and 180
// us for the exponents; now 15 us for both.
constexpr int kLogSumLanes = 1024, kLogSumChunk = 4096;

static __global__ __launch_bounds__(kLogSumLanes) void logsum_kernel(const double *util, const uint16_t *mask,
                                                                     int first, int n_used, int R, int rate_term,
                                                                     const int *xe, const int *ye, const int *ze,
                                                                     double *out) {
  __shared__ double v[kLogSumChunk];
  __shared__ long long sums[kLogSumLanes / 64][4];  // masked sites, exponent sums
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  long long used = 0, tx = 0, ty = 0, tz = 0;
  double ll = 0.0;  // in the first wave
  for (int c0 = 0; c0 < n_used; c0 += kLogSumChunk) {
    const int n = min(kLogSumChunk, n_used - c0), n_pad = (n + 63) & ~63;
    for (int i = threadIdx.x; i < n_pad; i += blockDim.x) {
      const int site = first + c0 + i;
      const bool in = i < n && (!mask || mask[site]);
      v[i] = in ? cr::log(util[c0 + i]) : 0.0;
      if (in) {
        used++;
        if (xe) { tx += xe[site]; ty += ye[site]; }
        if (ze) tz += ze[site];
      }
    }
    __syncthreads();
    if (wave == 0) ll = wave_sequential_sum(v, n, nullptr, ll);
    __syncthreads();
  }
  used = wave_sum_ll(used);
  tx = wave_sum_ll(tx);
  ty = wave_sum_ll(ty);
  tz = wave_sum_ll(tz);
  if (lane == 0) {
    sums[wave][0] = used;
    sums[wave][1] = tx;
    sums[wave][2] = ty;
    sums[wave][3] = tz;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < (int)(blockDim.x >> 6); w++) {
    used += sums[w][0];
    tx += sums[w][1];
    ty += sums[w][2];
    tz += sums[w][3];
  }
  if (rate_term) ll -= ((double)(float)used) * cr::log((double)(float)R);
  if (xe) ll = ll + PP_LOG2 * (ze ? ((double)tx + (double)ty) + (double)tz : (double)tx + (double)ty);
  *out = ll;
}

// The two kernels in order on a stream: util[0 .. n_used) and *out.
static inline void launch_logsum(hipStream_t st, double *util, const double *statd, const double *x, const double *y,
                                 const double *z, const uint16_t *mask, int first, int n_used, int R, int N, int S,
                                 int rate_term, const int *xe, const int *ye, const int *ze, double *out) {
  if (n_used > 0) {
    const auto k = S == 4 ? &util_kernel<4> : S == 20 ? &util_kernel<20> : &util_kernel<0>;
    hipLaunchKernelGGL(k, dim3((n_used + 63) / 64), dim3(64), 0, st, util, statd, x, y, z, mask, first, n_used, R, N,
                       S);
  }
  hipLaunchKernelGGL(logsum_kernel, dim3(1), dim3(kLogSumLanes), 0, st, util, mask, first, n_used, R, rate_term, xe,
                     ye, ze, out);
}

}  // namespace pp
