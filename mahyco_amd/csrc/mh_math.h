// mh_math.h -- arithmetic helpers shared by the HIP kernels and their host-side checks.
//
// mh_pow_third(x): x raised to the double nearest 1/3, correctly rounded.
//   MaHyCo's characteristic length is std::pow(V, 1./3.) (MahycoModule.cc:1219).  The
//   exponent fl(1/3) = 1/3 - d with d = 2^-54/3 ~ 1.85e-17, so
//       x^fl(1/3) = cbrt(x) * exp(-d ln x) = cbrt(x) * (1 - d ln x) + O(d^2 ln^2 x).
//   cbrt(x) is taken to double-double precision by one Newton step whose residual
//   x - c^3 is formed exactly with fma-based two-products; the d ln x term is ~1e-15
//   relative, so a plain-double log is ample.  The sum is rounded once, which yields the
//   correctly rounded power unless the exact value lies within ~1e-30 relative of a
//   rounding midpoint.  The same code on host and device gives the same bits even when
//   the library cbrt/log differ by an ulp.
// mh_pow_half(x): sqrt(x), the correctly rounded x^0.5 (pow(V, 0.5) in 2D).
#ifndef MH_MATH_H
#define MH_MATH_H

#include <cmath>

#ifdef __HIPCC__
#define MH_HD __host__ __device__ __forceinline__
#else
#define MH_HD inline
#endif

MH_HD double mh_pow_third(double x) {
  if (!(x > 0.0) || !std::isfinite(x)) return std::pow(x, 1.0 / 3.0);
  const double d = 1.8503717077085942e-17;  // 1/3 - fl(1/3) = 2^-54 / 3
  double c = std::cbrt(x);
  // c^3 = c2h*c + c2l*c, with c2h + c2l = c*c exactly
  double c2h = c * c;
  double c2l = std::fma(c, c, -c2h);
  double c3h = c2h * c;
  double c3l = std::fma(c2h, c, -c3h);
  double r = (x - c3h) - (c3l + c2l * c);  // x - c^3, accurate to ~2^-100 relative
  double lo = r / (3.0 * c2h);
  double corr = -d * std::log(x) * c;
  return c + (lo + corr);
}

MH_HD double mh_pow_half(double x) { return std::sqrt(x); }

// Several quotients a / b of one denominator: y = 1 / b is formed once (rounded to nearest), and
// each quotient takes q = a y, the remainder e = a - b q by one fma and q + e y by another -- the
// last steps of the division sequence itself, so each is the correctly rounded a / b, in 6
// instructions instead of 11, one of them a quarter-rate reciprocal.  Those steps hold while
// nothing leaves the normal range: a remainder that is not a number, infinite or subnormal
// (zero or infinite b, NaN, overflow) or an a below 2^-950, whose remainder may round to 0,
// sets `bad`, and the caller forms that group of quotients again by division.  (An advected
// bubble leaves densities down to 2^-1074 behind, so such operands do occur.)  mh_denom also rules out
// a b above 2^70: with both bounds q is no smaller than 2^-1020, where a subnormal quotient may lie
// at a tie that q + e y misses.  The bound is b's because a second one on every quotient costs 4 % of
// the sweeps, and a's is not higher because what moves ahead of a wave falls through all magnitudes
// (at 2^-520 2.5 % of a blast's dual sweeps).
struct MhRecip {
  double b, y;
  bool bad;  // y itself is outside the normal range
};
MH_HD bool mh_unsafe(double e) {  // NaN, infinite or subnormal
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_class(e, 0x297);
#else
  const int c = std::fpclassify(e);
  return c != FP_NORMAL && c != FP_ZERO;
#endif
}
MH_HD bool mh_tiny(double a) { return std::fabs(a) < 0x1p-950 && a != 0.; }
MH_HD MhRecip mh_recip(double b) {
  MhRecip r;
  r.b = b;
  r.y = 1.0 / b;
  r.bad = mh_unsafe(r.y);
  return r;
}
// the denominator of a group of quotients; where it is bad they are formed by division
MH_HD MhRecip mh_denom(double b) {
  MhRecip r = mh_recip(b);
  r.bad |= std::fabs(b) > 0x1p70;
  return r;
}
MH_HD double mh_div(double a, const MhRecip& r, bool& bad) {
  const double q = a * r.y;
  const double e = std::fma(-r.b, q, a);
  bad |= mh_unsafe(e) | mh_tiny(a);
  return std::fma(e, r.y, q);
}
// One quotient, formed again by division where it has to be.  mh_quot has the bits of a / b; a zero of
// mh_ratio, as one of mh_div, may have either sign (the remainder of -0 is +0): for values that only
// enter sums from 0, as those of the sweeps do.
MH_HD double mh_ratio(double a, const MhRecip& r) {
  bool bad = r.bad;
  double q = mh_div(a, r, bad);
  if (__builtin_expect(bad, 0)) q = a / r.b;
  return q;
}
MH_HD double mh_quot(double a, const MhRecip& r) {
  bool bad = r.bad;
  double q = std::copysign(mh_div(a, r, bad), a * r.y);
  if (__builtin_expect(bad, 0)) q = a / r.b;
  return q;
}

#endif
