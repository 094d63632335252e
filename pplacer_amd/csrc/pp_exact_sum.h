// The stub's sequential log sum (linear_c.c:416-419), 0 + v[0] + v[1] + ...
// + v[n-1] with one rounding per term in site order, bit for bit, computed by
// a whole wave instead of one lane.
//
// Why a wave can do it: let s_k be the sequential partial sums and u_E =
// 2^(E-53) the spacing of doubles in the binade [2^(E-1), 2^E) (frexp
// exponent E).  While the partial sums stay in one binade they are multiples
// of u_E, and adding v_k rounds to s_{k-1} + rint(v_k / u_E) u_E unless v_k /
// u_E is exactly halfway between integers (a tie goes to even and so depends
// on s_{k-1}).  A run of such additions moves any starting value of the
// binade by the same multiple of u_E.
//
// So the terms are split into 64 contiguous blocks of B = ceil(n / 64), one a
// lane, and
//  1. a DPP scan of block sums gives each lane an approximate partial sum p
//     before its block, within delta = (4n + 256) 2^-53 sum|v| of the true one
//     (recursive summation error bounds, doubled);
//  2. every lane runs the real, rounding additions of its block from p.  The
//     block is "clean" if its terms are <= 0, none of the additions is a tie,
//     and p and the end value, each moved delta outwards, lie in one binade:
//     then the true partial sums lie in it too, and the block moves the true
//     sum by exactly (end - p);
//  3. the moves of consecutive clean blocks add up exactly (multiples of one
//     u_E, less than 2^53 of them), in any order: a DPP scan that restarts at
//     the other blocks;
//  4. the other blocks (the first, those that change the binade or hold a
//     tie; about 8 at 300 terms) are run again in order from the true sum.
//     Whatever a block holds (mixed signs, infinities, NaN), that is the
//     sequential sum itself, so only how many blocks are run again depends on
//     the terms.
//
// What it costs: B dependent additions twice, two scans of 6 steps, and B
// additions and two lane reads for each block run again.  On one wave: 1,700
// cycles at 300 terms against 5,200 for the chain of one lane (17 cycles a
// term), 1,000 against 1,900 at 100.
#pragma once

#include <hip/hip_runtime.h>

#include "pp_device.h"

namespace pp {

// Longest sum the wave takes; longer ones go to the one-lane chain.
constexpr int kSeqSumWaveMax = 4096;

// s + v[0] + v[1] + ... + v[n-1], one lane.  A dependent chain, so it is fed
// from LDS two blocks of eight ahead: the loads of one block are in flight
// while the previous block is added.
__device__ __forceinline__ double ordered_sum(const double *v, int n, double s = 0.0) {
  double a[8], b[8];
#pragma unroll
  for (int j = 0; j < 8; j++) a[j] = j < n ? v[j] : 0.0;
#pragma unroll
  for (int j = 0; j < 8; j++) b[j] = 8 + j < n ? v[8 + j] : 0.0;
  int i = 0;
  for (; i + 32 <= n; i += 16) {  // a = v[i..i+8), b = v[i+8..i+16), both in range
#pragma unroll
    for (int j = 0; j < 8; j++) s += a[j];
#pragma unroll
    for (int j = 0; j < 8; j++) a[j] = v[i + 16 + j];
#pragma unroll
    for (int j = 0; j < 8; j++) s += b[j];
#pragma unroll
    for (int j = 0; j < 8; j++) b[j] = v[i + 24 + j];
  }
  // fewer than 32 left: a and b hold v[i .. i+16) where in range
#pragma unroll
  for (int j = 0; j < 8; j++)
    if (i + j < n) s += a[j];
#pragma unroll
  for (int j = 0; j < 8; j++)
    if (i + 8 + j < n) s += b[j];
  for (i += 16; i < n; i++) s += v[i];
  return s;
}

// v from the lane CTRL selects; lanes whose row ROWMASK leaves out, or whose
// source lane falls outside the row, get 0.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ int dpp_i32_or0(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWMASK, 0xF, false);
}
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_f64_or0(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)dpp_i32_or0<CTRL, ROWMASK>((int)(unsigned)b);
  const unsigned hi = (unsigned)dpp_i32_or0<CTRL, ROWMASK>((int)(unsigned)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Inclusive prefix sums over the wave (all 64 lanes active): shifts by 1, 2,
// 4 and 8 within each row of 16, then row 0's total into row 1 and row 2's
// into row 3 (row_bcast:15), then rows 0-1's total into rows 2 and 3
// (row_bcast:31).
__device__ __forceinline__ int wave_scan_i32(int v) {
  v += dpp_i32_or0<0x111, 0xF>(v);
  v += dpp_i32_or0<0x112, 0xF>(v);
  v += dpp_i32_or0<0x114, 0xF>(v);
  v += dpp_i32_or0<0x118, 0xF>(v);
  v += dpp_i32_or0<0x142, 0xA>(v);
  v += dpp_i32_or0<0x143, 0xC>(v);
  return v;
}
__device__ __forceinline__ double wave_scan_f64(double v) {
  v += dpp_f64_or0<0x111, 0xF>(v);
  v += dpp_f64_or0<0x112, 0xF>(v);
  v += dpp_f64_or0<0x114, 0xF>(v);
  v += dpp_f64_or0<0x118, 0xF>(v);
  v += dpp_f64_or0<0x142, 0xA>(v);
  v += dpp_f64_or0<0x143, 0xC>(v);
  return v;
}

// Inclusive prefix sums that restart at every lane set in `starts` (bit 0
// set): lane l gets the sum from its run's first lane, the highest set bit of
// starts up to l.  The steps of wave_scan_f64; a step's source is taken where
// it lies in the lane's own run.
__device__ __forceinline__ double wave_run_scan_f64(double v, unsigned long long starts) {
  const int lane = fresh_lane();
  const int first = 63 - __builtin_clzll(starts & (~0ull >> (63 - lane)));
  const int back = lane - first;  // lanes of the run before this one
  double t = dpp_f64_or0<0x111, 0xF>(v);
  v += back >= 1 ? t : 0.0;
  t = dpp_f64_or0<0x112, 0xF>(v);
  v += back >= 2 ? t : 0.0;
  t = dpp_f64_or0<0x114, 0xF>(v);
  v += back >= 4 ? t : 0.0;
  t = dpp_f64_or0<0x118, 0xF>(v);
  v += back >= 8 ? t : 0.0;
  t = dpp_f64_or0<0x142, 0xA>(v);
  v += first < (lane & 0x30) ? t : 0.0;  // the row's run comes out of the row before
  t = dpp_f64_or0<0x143, 0xC>(v);
  v += first < 32 ? t : 0.0;
  return v;
}

// The terms of a lane's block, B (wave-uniform) of them from v + lane B: in
// registers when the block has at most CAP, else read from LDS as they are
// needed.
template <int CAP>
struct SeqSumBlock {
  const double *v;
  int B;
  double x[CAP > 0 ? CAP : 1];
  __device__ __forceinline__ void load(const double *v0, int b) {
    v = v0 + fresh_lane() * b;
    B = b;
#pragma unroll
    for (int j = 0; j < CAP; j++) x[j] = v[j < B ? j : 0];
  }
  template <class F>
  __device__ __forceinline__ void each(F &&f) const {
    if constexpr (CAP > 0) {
#pragma unroll
      for (int j = 0; j < CAP; j++)
        if (j < B) f(x[j]);
    } else {
      int j = 0;
#pragma unroll 1
      for (; j + 8 <= B; j += 8) {
        double y[8];
#pragma unroll
        for (int i = 0; i < 8; i++) y[i] = v[j + i];
#pragma unroll
        for (int i = 0; i < 8; i++) f(y[i]);
      }
#pragma unroll 1
      for (; j < B; j++) f(v[j]);
    }
  }
};

template <int CAP>
__device__ __forceinline__ double wave_sequential_sum_of(const double *v, int n, int B, int *n_events, double start) {
  SeqSumBlock<CAP> blk;
  blk.load(v, B);
  double a = 0.0, top = -INFINITY;
  blk.each([&](double x) {
    a += x;
    top = fmax(top, x);
  });
  const double incl = wave_scan_f64(a);
  const bool inner = fresh_lane() != 0;
  const double p = inner ? start + (incl - a) : start;  // approximate partial sum before the block
  double Q = -(start + readlane_f64(incl, 63));
  if (wave_true(!(top <= 0.0))) {  // not every term is <= 0
    double q = 0.0;
    blk.each([&](double x) { q += fabs(x); });
    Q = wave_sum(q) + fabs(start);
  }
  const double delta = (4.0 * n + 256.0) * 0x1p-53 * Q;
  double s = p;
  bool tie = false;
  const double half_u = __builtin_amdgcn_ldexp(1.0, __builtin_amdgcn_frexp_exp(p) - 54);
  blk.each([&](double x) {
    const double t = s + x;
    tie |= fabs(x - (t - s)) == half_u;  // the addition's exact error, in a clean block
    s = t;
  });
  const bool clean = inner & (top <= 0.0) & (start <= 0.0) & !tie & (Q <= 0x1p+996) & (Q >= 0x1p-900) & (fabs(p) > delta) &
                     (__builtin_amdgcn_frexp_exp(fabs(p) - delta) == __builtin_amdgcn_frexp_exp(fabs(s) + delta));
  const unsigned long long again = __builtin_amdgcn_ballot_w64(!clean) | 1ull;
  const double move = wave_run_scan_f64(clean ? s - p : 0.0, again);
  if (n_events) *n_events = __builtin_popcountll(again);
  double sum = readlane_f64(s, 0);  // block 0 started from the true sum itself
  const double before = dpp_f64_or0<0x138, 0xF>(move);  // of the run that ends before the lane
#pragma unroll 1
  for (unsigned long long rest = again & ~1ull; rest; rest &= rest - 1) {
    double t = sum + before;  // every lane, only lane j's is the sum
    blk.each([&](double x) { t += x; });
    sum = readlane_f64(t, __builtin_ctzll(rest));
  }
  return sum + readlane_f64(move, 63);
}

// Sequential sum of v[0..n) (LDS, n wave-uniform), the same value in every
// lane; call with the whole wave active.  v holds 64 ceil(n / 64) doubles,
// those past n being 0.0 (adding them changes no sum).  The sum goes on from
// `start` (a longer sum in pieces; not -0.0).  *n_events (when given) receives
// the number of blocks added from the true sum, or -1 where the one-lane chain
// ran.
__device__ __forceinline__ double wave_sequential_sum(const double *v, int n, int *n_events = nullptr,
                                                      double start = 0.0) {
  if (n <= 0) {
    if (n_events) *n_events = 0;
    return start;
  }
  if (n <= 256) return wave_sequential_sum_of<4>(v, n, (n + 63) >> 6, n_events, start);
  if (n <= 512) return wave_sequential_sum_of<8>(v, n, (n + 63) >> 6, n_events, start);
  if (n <= kSeqSumWaveMax) return wave_sequential_sum_of<0>(v, n, (n + 63) >> 6, n_events, start);
  if (n_events) *n_events = -1;
  double s = 0.0;
  if ((threadIdx.x & 63) == 0) s = ordered_sum(v, n, start);
  return readlane_f64(s, 0);
}

}  // namespace pp
