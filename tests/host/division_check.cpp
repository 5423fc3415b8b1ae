// Host check of the shared-denominator division and the one-division limiters (mh_math.h,
// mh_geom.h) against the plain forms.  Reads pairs of doubles (hexadecimal bit patterns) on
// stdin; prints the pairs read and the mismatches of the division (quotients not flagged, or
// flagged quotients of ordinary operands) and of the limited gradients.
#include <cinttypes>
#include <cstdio>
#include <cstring>
#include "../../mahyco_amd/csrc/mh_geom.h"

static double from_bits(uint64_t u) { double v; std::memcpy(&v, &u, 8); return v; }
static bool same(double a, double b) { return a == b || (a != a && b != b); }

template <int LIM>
static double two_sided(double gb, double gf) {
  double g = 0.;
  if (gb != 0.) g += 0.5 * (mh_flux_limiter(LIM, gf / gb) * gb);
  if (gf != 0.) g += 0.5 * (mh_flux_limiter(LIM, gb / gf) * gf);
  return g;
}
static bool ordinary(double v) { return v == 0. || (std::fabs(v) > 1e-140 && std::fabs(v) < 1e140); }

int main() {
  long pairs = 0, div = 0, lim = 0;
  uint64_t a, b;
  while (std::scanf("%" SCNx64 " %" SCNx64, &a, &b) == 2) {
    const double x = from_bits(a), y = from_bits(b);
    const MhRecip r = mh_recip(y);
    bool bad = r.bad;
    const double q = mh_div(x, r, bad);
    if (!same(mh_quot(x, r), x / y)) ++div;
    if (!bad && !same(q, x / y)) ++div;
    if (bad && ordinary(x) && ordinary(y) && y != 0.) ++div;
    if (!same(mh_limited_gradient<0>(0, x, y), two_sided<0>(x, y))) ++lim;
    if (!same(mh_limited_gradient<1>(1, x, y), two_sided<1>(x, y))) ++lim;
    if (!same(mh_limited_gradient<2>(2, x, y), two_sided<2>(x, y))) ++lim;
    if (!same(mh_limited_gradient<3>(3, x, y), two_sided<3>(x, y))) ++lim;
    // the dual sweeps' rounding, (1/2 phi) g
    double g = 0.;
    if (x != 0.) g += 0.5 * mh_flux_limiter(1, y / x) * x;
    if (y != 0.) g += 0.5 * mh_flux_limiter(1, x / y) * y;
    if (!same(mh_limited_gradient<1, true>(1, x, y), g)) ++lim;
    g = 0.;
    if (x != 0.) g += 0.5 * mh_flux_limiter(0, y / x) * x;
    if (y != 0.) g += 0.5 * mh_flux_limiter(0, x / y) * y;
    if (!same(mh_limited_gradient<0, true>(0, x, y), g)) ++lim;
    ++pairs;
  }
  std::printf("%ld %ld %ld\n", pairs, div, lim);
  return 0;
}
