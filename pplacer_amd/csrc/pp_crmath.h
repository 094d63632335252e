// Correctly rounded FP64 exp and log, for the FP64 form's transition
// matrices and site logs.
//
// The C stubs call the host libm (glibc), whose exp and log return the
// correctly rounded result in all but a tiny fraction of cases; the device's
// library routines are faithful (within one ulp) but differ from the
// correctly rounded value on a few percent of exp and a fraction of a
// percent of log arguments.  Each such ulp can flip a Brent comparison at a
// flat optimum.  These routines return the correctly rounded result, so the
// device agrees with the stubs' libm wherever that libm rounds correctly.
//
// Method (Ziv's strategy, table-driven, own constants from
// gen_crmath_tables.py):
// * exp: x = k ln2/128 + r, |r| <= ln2/256 (+ rounding), exp(x) =
//   2^(k >> 7) * 2^((k & 127)/128) * exp(r), the table entry a double-double;
//   r is reduced in double-double (ln2/128 = C1 + C2 + C3, k*C1 exact), and
//   exp(r) = 1 + r + r^2/2 + r^3 q(r) with r^2 split exactly.  Relative error
//   below 2^-77.
// * log: x = 2^e m, m in [0.75, 1.5); m's interval j of width 1/128 gives
//   u = m inv[j] - 1, |u| < 2^-6, and
//   log x = e ln2 + L[j] + log1p(u) with L[j] = -log(inv[j]) a double-double;
//   inv[j] (1/(interval centre) rounded to 8 significant bits) is formed
//   arithmetically, so that u = m inv[j] - 1 (as an exact double-double) is
//   ready while L[j] loads; log1p(u) = u - u^2/2 + u^3 Q(u) with u^2 kept
//   exactly.  Absolute error below 2^-51 |u^3| + 2^-73 |log x|.
// * The double-double result (h, l) is rounded to nearest and accepted when
//   h + l +/- d round alike (d = 2^-74 |h| for exp, 2^-51 |u^3| + 2^-71 |h|
//   for log, above the error bounds); otherwise (the value lies that close to a
//   rounding boundary) it is recomputed in double-double throughout (error
//   about 2^-100) and rounded.  Counted on 2 10^7 arguments each, in 10^5: exp
//   0.1; log none below 1/e, 1 on [0.5, 1), 9 on [0.98, 1) and 24 on
//   [1 - 2^-7, 1 - 2^-8], where u is largest and no e ln2 or L outweighs it.
// * Outside the fast range -- exp of x <= -708.3 (subnormal results) or
//   >= 709.7, log of zero, negatives, subnormals, infinities, NaN -- the
//   library routine answers.
// Every operation is a separately rounded IEEE operation or an fma: the
// library is built with -ffp-contract=off, so the error-free transformations
// below hold on the host and the device alike.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define PP_CR_FN __device__ __forceinline__
#define PP_CR_SLOW __device__ __attribute__((noinline))
#define PP_CR_TAB static __constant__ const
#else
#define PP_CR_FN static inline
#define PP_CR_SLOW static
#define PP_CR_TAB static const
#endif

// The coefficients the fast paths name one by one are constant expressions:
// they become literals, which a kernel short of registers makes again where it
// needs them.  (Loaded from memory they were hoisted out of the probe loops
// and spilled.)
#define PP_CR_CST static constexpr

#include "pp_crmath_tables.h"

namespace pp {
namespace cr {

struct DD {
  double hi, lo;
};

// A coefficient made where it is used: on the device a pair of scalar moves
// that stays inside the loop it is written in.  Left to itself the compiler
// keeps such constants in vector registers across a kernel's probe loop, and
// spills them.
PP_CR_FN double lit(double c) {
#if defined(__HIPCC__) && defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(c));
#endif
  return c;
}

PP_CR_FN DD two_sum(double a, double b) {
  const double s = a + b, bb = s - a;
  return {s, (a - (s - bb)) + (b - bb)};
}
// |a| >= |b| (or a == 0)
PP_CR_FN DD fast_two_sum(double a, double b) {
  const double s = a + b;
  return {s, b - (s - a)};
}
PP_CR_FN DD two_prod(double a, double b) {
  const double p = a * b;
  return {p, fma(a, b, -p)};
}
PP_CR_FN DD dd_add(DD a, DD b) {
  DD s = two_sum(a.hi, b.hi);
  const DD t = two_sum(a.lo, b.lo);
  s = fast_two_sum(s.hi, s.lo + t.hi);
  return fast_two_sum(s.hi, s.lo + t.lo);
}
PP_CR_FN DD dd_mul(DD a, DD b) {
  const DD p = two_prod(a.hi, b.hi);
  return fast_two_sum(p.hi, p.lo + (a.hi * b.lo + a.lo * b.hi));
}
PP_CR_FN DD dd_mul_d(DD a, double b) {
  const DD p = two_prod(a.hi, b);
  return fast_two_sum(p.hi, p.lo + a.lo * b);
}

// h + l rounded to nearest; ok when every value within d of h + l rounds to
// the same double (rounding is monotone, so the two ends decide).
PP_CR_FN double round_checked(double h, double l, double d, bool &ok) {
  const double r = h + l;
  ok = (h + (l + d)) == r && (h + (l - d)) == r;
  return r;
}

// x = k ln2/128 + r with r a double-double: k C1 is exact and x - k C1 exact
// (Sterbenz)
PP_CR_FN DD exp_reduce(double x, double kf) {
  const double r1 = x - kf * pp_cr_exp_c[1];
  const DD p2 = two_prod(kf, pp_cr_exp_c[2]);
  const DD r = two_sum(r1, -p2.hi);
  return fast_two_sum(r.hi, (r.lo - p2.lo) - kf * pp_cr_exp_c[3]);
}

// exp(x) where the fast path cannot decide: the library's outside the fast
// range, else exp(r) * T in double-double, Horner over 1/k!, k = 13..0.  A
// call with one argument: nothing of the fast path has to live across it.
PP_CR_SLOW double exp_slow(double x) {
  if (!(x > -708.3 && x < 709.7)) return ::exp(x);
  const double kf = rint(x * pp_cr_exp_c[0]);
  const int k = (int)kf, j = k & 127, m = (k - j) >> 7;
  const DD r = exp_reduce(x, kf), t = {pp_cr_exp_t[2 * j], pp_cr_exp_t[2 * j + 1]};
  DD p = {pp_cr_exp_pdd[26], pp_cr_exp_pdd[27]};
#if defined(__HIPCC__)
#pragma unroll 1
#endif
  for (int i = 12; i >= 0; i--) p = dd_add(dd_mul(p, r), DD{pp_cr_exp_pdd[2 * i], pp_cr_exp_pdd[2 * i + 1]});
  const DD y = dd_mul(p, t);
  bool ok;
  return ldexp(round_checked(y.hi, y.lo, 0x1p-100 * fabs(y.hi), ok), m);
}

// The library's exp and log answer outside the fast range, but only inside
// the slow path's call: inlined here as the other side of a range check, the
// compiler evaluated them for every argument, spills included (a site's log
// in the 4-state kernels: 4,500 -> 1,800 cycles on one wave).
PP_CR_FN double exp(double x) {
  const bool in = x > -708.3 && x < 709.7;
  const double kf = rint(x * pp_cr_exp_c[0]);
  const int k = (int)kf, j = k & 127, m = (k - j) >> 7;  // k = 128 m + j
  const DD t = {pp_cr_exp_t[2 * j], pp_cr_exp_t[2 * j + 1]};
  const DD r = exp_reduce(x, kf);
  // exp(r) - 1 = rh + sq.hi/2 + tail, sq = rh^2 exactly
  const double rh = r.hi, rl = r.lo;
  const DD sq = two_prod(rh, rh);
  const double *c = pp_cr_exp_p;
  const double q = fma(rh, fma(rh, fma(rh, fma(rh, lit(c[7]), lit(c[6])), lit(c[5])), lit(c[4])), lit(c[3]));
  const double tail = 0.5 * sq.lo + (sq.hi * rh) * q + (rl + rl * rh);
  const double half_sq = 0.5 * sq.hi;
  // T (1 + E) = t.hi + t.hi rh + t.hi sq/2 + (t.hi tail + t.lo + t.lo E)
  const DD a = two_prod(t.hi, rh), b = two_prod(t.hi, half_sq);
  const double tl = t.hi * tail + t.lo + t.lo * (rh + half_sq);
  const DD s1 = fast_two_sum(t.hi, a.hi), s2 = fast_two_sum(s1.hi, b.hi);
  const DD y = fast_two_sum(s2.hi, (s1.lo + s2.lo) + ((a.lo + b.lo) + tl));
  bool ok;
  const double res = ldexp(round_checked(y.hi, y.lo, 0x1p-74 * fabs(y.hi), ok), m);
  return in && ok ? res : exp_slow(x);
}

// Reduction of x = 2^e m, m in [0.75, 1.5): interval j, and u + ul = m inv[j]
// - 1 exactly.
struct LogRed {
  int j;
  double e, u, ul;
};
PP_CR_FN LogRed log_reduce(double x) {
  LogRed g;
  int e;
  const double m0 = frexp(x, &e);
  const bool low = m0 < 0.75;
  const double m = low ? m0 + m0 : m0;
  g.e = (double)(low ? e - 1 : e);
  int j = (int)((m - 0.75) * 128.);  // m - 0.75 exact
  j = j < 0 ? 0 : j > 95 ? 95 : j;   // (arguments out of range stay in the table)
  g.j = j;
  // inv[j]: 1/(interval centre) rounded to 8 significant bits; 1 next to 1.
  // No 1/centre lies within 2^-13 of a rounding boundary, so an approximate
  // single-precision reciprocal gives the same bits as the exact one.
#if defined(__HIPCC__) && defined(__HIP_DEVICE_COMPILE__)
  const float q = __builtin_amdgcn_rcpf(0.75f + ((float)j + 0.5f) * 0.0078125f);
#else
  const float q = 1.f / (0.75f + ((float)j + 0.5f) * 0.0078125f);
#endif
  const float up = q < 1.f ? 256.f : 128.f, down = q < 1.f ? 0x1p-8f : 0x1p-7f;
  const double inv = (j == 31 || j == 32) ? 1.f : rintf(q * up) * down;
  // p - 1 is exact (p is within 2^-6 of 1), and zero or larger than the error
  const double p = m * inv;
  const DD uu = fast_two_sum(p - 1., fma(m, inv, -p));
  g.u = uu.hi;
  g.ul = uu.lo;
  return g;
}

// log(x) where the fast path cannot decide: the library's outside the fast
// range, else e ln2 + L + log1p(u) in double-double, Horner over
// (-1)^(k+1)/k, k = 18..1 (a call, as exp_slow)
PP_CR_SLOW double log_slow(double x) {
  if (!(x >= 0x1p-1022 && x < INFINITY)) return ::log(x);
  const LogRed g = log_reduce(x);
  const DD u = {g.u, g.ul}, l = {pp_cr_log_l[2 * g.j], pp_cr_log_l[2 * g.j + 1]};
  DD p = {pp_cr_log_pdd[34], pp_cr_log_pdd[35]};
#if defined(__HIPCC__)
#pragma unroll 1
#endif
  for (int k = 16; k >= 0; k--) p = dd_add(dd_mul(p, u), DD{pp_cr_log_pdd[2 * k], pp_cr_log_pdd[2 * k + 1]});
  p = dd_mul(p, u);
  const DD e2 = two_prod(g.e, pp_cr_ln2[1]);
  DD en = fast_two_sum(g.e * pp_cr_ln2[0], e2.hi);  // e hi is exact
  en = fast_two_sum(en.hi, en.lo + (e2.lo + g.e * pp_cr_ln2[2]));
  const DD y = dd_add(dd_add(en, l), p);
  bool ok;
  return round_checked(y.hi, y.lo, 0x1p-100 * fabs(y.hi), ok);
}

PP_CR_FN double log(double x) {
  const bool in = x >= 0x1p-1022 && x < INFINITY;
  const LogRed g = log_reduce(x);
  const DD l = {pp_cr_log_l[2 * g.j], pp_cr_log_l[2 * g.j + 1]};
  const double u = g.u;
  const DD u2 = two_prod(u, u);
  // r = u^3 Q(u), Q(u) = sum_{k=2..12} c_k u^(k-2) by Estrin's scheme, each
  // operation correct to 2^-53: r is off by less than 2^-51 |u^3| (with the
  // additions that take it up), the terms past u^13 by less than 2^-81
  const double *c = pp_cr_log_p;
  const double w2 = u2.hi, w4 = w2 * w2, u3 = w2 * u;
  const double q0 = fma(w2, fma(u, lit(c[5]), lit(c[4])), fma(u, lit(c[3]), lit(c[2])));
  const double q1 = fma(w2, fma(u, lit(c[9]), lit(c[8])), fma(u, lit(c[7]), lit(c[6])));
  const double q2 = fma(w2, lit(c[12]), fma(u, lit(c[11]), lit(c[10])));
  const double r = u3 * fma(w4, fma(w4, q2, q1), q0);
  // e ln2 + L + u - u^2/2 + r: |e ln2| >= ln2 > |L|, |L| >= 2^-8 or L = 0
  // (and then |u| >= 2^-53 |u^2|): only u's term needs a two_sum
  DD s = fast_two_sum(g.e * pp_cr_ln2[0], l.hi);
  double lo = s.lo;
  s = two_sum(s.hi, u);
  lo += s.lo;
  s = fast_two_sum(s.hi, -0.5 * w2);
  lo += s.lo;
  // ul / (1 + u) for the part of u past one double
  lo += (fma(g.e, pp_cr_ln2[1], l.lo) - 0.5 * u2.lo) + (fma(-g.ul, u, g.ul) + r);
  const DD y = fast_two_sum(s.hi, lo);
  bool ok;
  const double res = round_checked(y.hi, y.lo, fma(fabs(u3), 0x1p-51, 0x1p-71 * fabs(y.hi)), ok);
  return in && ok ? res : log_slow(x);
}

}  // namespace cr
}  // namespace pp
