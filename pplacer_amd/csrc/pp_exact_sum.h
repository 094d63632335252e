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
// So every lane adds the first 32 terms one by one, and the others are split
// into 64 contiguous blocks, one a lane, of 4, 8, 16 or 24 terms:
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
//     tie; about 5 at 300 terms) are run again in order from the true sum.
//     Whatever a block holds (mixed signs, infinities, NaN), that is the
//     sequential sum itself, so only how many blocks are run again depends on
//     the terms.
//
// What bounds it is the length of the dependent chain (an FP64 addition 8
// cycles, a lane read into the next addition 32): two scans of 6 steps, the
// blocks' additions twice and again for each block run again.  In the engine's
// control wave: 2,150 cycles at 209 terms and 4,430 at 1,080 beside another
// workgroup; 2,790 and 10,280 without the head, with blocks of ceil(n / 64)
// terms read from LDS beyond 512; 17 cycles a term for the chain of one lane.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

#include "pp_device.h"

namespace pp {

// Longest sum the wave takes; longer ones go to the one-lane chain.
constexpr int kSeqSumWaveMax = 4096;
constexpr int kSeqSumHead = 32;

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
  // with whole rows the hardware's own zero for a source outside the row
  // (bound_ctrl) saves setting the result first
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWMASK, 0xF, ROWMASK == 0xF);
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
// between(): called before and after each of the six steps, for work that the
// steps' latency covers.
template <class F>
__device__ __forceinline__ double wave_scan_f64(double v, F &&between) {
  between();
  v += dpp_f64_or0<0x111, 0xF>(v);
  between();
  v += dpp_f64_or0<0x112, 0xF>(v);
  between();
  v += dpp_f64_or0<0x114, 0xF>(v);
  between();
  v += dpp_f64_or0<0x118, 0xF>(v);
  between();
  v += dpp_f64_or0<0x142, 0xA>(v);
  between();
  v += dpp_f64_or0<0x143, 0xC>(v);
  between();
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

// The terms of a lane's block: CAP of them from v + first, in registers, 0.0
// for a lane past the terms; CAP = 0: B (wave-uniform) of them, read from LDS
// as they are needed.
template <int CAP>
struct SeqSumBlock {
  double x[CAP > 0 ? CAP : 1];
  const double *v;
  int B, rest;  // CAP = 0: terms from v
  __device__ __forceinline__ void load(const double *terms, int n) {
    if constexpr (CAP > 0) {
      const int at = fresh_lane() * CAP;
#pragma unroll
      for (int j = 0; j < CAP; j++) x[j] = 0.0;
      if (at < n)
#pragma unroll
        for (int j = 0; j < CAP; j++) x[j] = terms[at + j];
    } else {
      B = (n + 63) >> 6;
      v = terms + fresh_lane() * B;
      rest = n - fresh_lane() * B;
    }
  }
  template <class F>
  __device__ __forceinline__ void each(F &&f) const {
    if constexpr (CAP > 0) {
#pragma unroll
      for (int j = 0; j < CAP; j++) f(x[j]);
    } else {
#pragma unroll 1
      for (int j = 0; j < B; j += 8) {
        double y[8];
#pragma unroll
        for (int i = 0; i < 8; i++) y[i] = j + i < B && j + i < rest ? v[j + i] : 0.0;
#pragma unroll
        for (int i = 0; i < 8; i++) f(y[i]);
      }
    }
  }
};

// head: the first terms, a multiple of 8, that every lane adds one by one.
// They hold about half of the binade changes and ties, and their chain runs in
// the shadow of the scan.
template <int CAP>
__device__ __forceinline__ double wave_sequential_sum_of(const double *v, int head, int n, int *n_events,
                                                         double start) {
  SeqSumBlock<CAP> blk;
  blk.load(v + head, n - head);
  // The block's loads first (after the head's they cost 400 reads with -p 1.7%),
  // the head's eight ahead, its additions among those of the blocks and the
  // scan's steps, as written (left to itself the compiler finished the scan
  // first and then waited for LDS at every eighth addition)
  double h = start, y[8];
#pragma unroll
  for (int j = 0; j < 8; j++) y[j] = v[j];
  double a = 0.0;
  double top = 0.0;
  blk.each([&](double x) {
    a += x;
    top = fmax(top, x);
  });
  const bool neg = top <= 0.0;
  int i = 0;
  const double incl = wave_scan_f64(a, [&] {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 5; j++, i++)
      if (i < kSeqSumHead) {
        h += y[i % 8];
        if (i + 8 < kSeqSumHead) y[i % 8] = v[i + 8];
      }
    __builtin_amdgcn_sched_barrier(0);
  });
#pragma unroll 1
  for (int k = kSeqSumHead; k < head; k += 8) {
#pragma unroll
    for (int j = 0; j < 8; j++) y[j] = v[k + j];
#pragma unroll
    for (int j = 0; j < 8; j++) h += y[j];
  }
  const bool inner = fresh_lane() != 0;
  const double p = inner ? h + (incl - a) : h;  // approximate partial sum before the block
  double Q = -(h + readlane_f64(incl, 63));
  if (wave_true(!neg)) {  // not every term is <= 0
    double q = 0.0;
    blk.each([&](double x) { q += fabs(x); });
    Q = wave_sum(q) + fabs(h);
  }
  const double delta = (4.0 * n + 256.0) * 0x1p-53 * Q;
  double s = p;
  double err = 0.0;  // the additions' largest exact error; half_u where one is a tie, no more in a clean block
  const double half_u = __builtin_amdgcn_ldexp(1.0, __builtin_amdgcn_frexp_exp(p) - 54);
  blk.each([&](double x) {
    const double t = s + x;
    err = fmax(err, fabs(x - (t - s)));
    s = t;
  });
  const bool clean = inner & neg & (h <= 0.0) & (err != half_u) & (Q <= 0x1p+996) & (Q >= 0x1p-900) & (fabs(p) > delta) &
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
// `start` (a longer sum in pieces; not -0.0).  NMAX bounds n where it is known.
// *n_events (when given) receives the number of blocks added from the true
// sum, or -1 where the one-lane chain ran.
//
// A block is the 4, 8, 16 or 24 terms that 64 lanes need to cover n (n up to
// 4,096: n / 64, from LDS).  The blocks end where v does: 4, 8 and 16 divide
// 64 less the head, and for 24 the head is as long as that takes.
template <int NMAX = INT_MAX>
__device__ __forceinline__ double wave_sequential_sum(const double *v, int n, int *n_events = nullptr,
                                                      double start = 0.0) {
  constexpr int H = kSeqSumHead;
  if (n <= 0) {
    if (n_events) *n_events = 0;
    return start;
  }
  if (NMAX <= H + 256 || n <= H + 256) return wave_sequential_sum_of<4>(v, H, n, n_events, start);
  if (NMAX <= H + 512 || n <= H + 512) return wave_sequential_sum_of<8>(v, H, n, n_events, start);
  if (NMAX <= H + 1024 || n <= H + 1024) return wave_sequential_sum_of<16>(v, H, n, n_events, start);
  if (n <= H + 1536) {
    const int m = ((n + 63) >> 6) % 3;  // 64 m' - head a multiple of 24
    return wave_sequential_sum_of<24>(v, m == 0 ? 48 : m == 1 ? 40 : 32, n, n_events, start);
  }
  if (n <= kSeqSumWaveMax) return wave_sequential_sum_of<0>(v, H, n, n_events, start);
  if (n_events) *n_events = -1;
  double s = 0.0;
  if ((threadIdx.x & 63) == 0) s = ordered_sum(v, n, start);
  return readlane_f64(s, 0);
}

}  // namespace pp
