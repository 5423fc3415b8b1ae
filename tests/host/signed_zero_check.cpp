// Host check of the shared-denominator quotients (mh_math.h) and the one-division limited gradients
// (mh_geom.h): mh_quot gives the bits of plain division, signs of zero included; mh_div where it is
// taken, and the gradients against the two-sided formula, but for the sign of a zero.  Reads pairs of
// doubles (hexadecimal bit patterns) on stdin; prints the pairs read and the mismatches of the quotients
// and of the gradients.  (A NaN matches any NaN.)
#include <cinttypes>
#include <cstdio>
#include <cstring>
#include "../../mahyco_amd/csrc/mh_geom.h"

static double from_bits(uint64_t u) { double v; std::memcpy(&v, &u, 8); return v; }
static uint64_t bits(double v) { uint64_t u; std::memcpy(&u, &v, 8); return u; }
static bool same(double a, double b) { return bits(a) == bits(b) || (a != a && b != b); }
static bool equal(double a, double b) { return a == b || (a != a && b != b); }

template <int LIM, bool DUAL>
static double two_sided(double gb, double gf) {
  auto term = [](double phi, double g) { return DUAL ? (0.5 * phi) * g : 0.5 * (phi * g); };
  double g = 0.;
  if (gb != 0.) g += term(mh_flux_limiter(LIM, gf / gb), gb);
  if (gf != 0.) g += term(mh_flux_limiter(LIM, gb / gf), gf);
  return g;
}
template <int LIM>
static bool gradient(double x, double y) {
  return equal(mh_limited_gradient<LIM>(LIM, x, y), two_sided<LIM, false>(x, y)) &&
         equal(mh_limited_gradient<LIM, true>(LIM, x, y), two_sided<LIM, true>(x, y));
}

int main() {
  long pairs = 0, div = 0, lim = 0;
  uint64_t a, b;
  while (std::scanf("%" SCNx64 " %" SCNx64, &a, &b) == 2) {
    const double x = from_bits(a), y = from_bits(b);
    div += !same(mh_quot(x, mh_denom(y)), x / y) + !equal(mh_ratio(x, mh_denom(y)), x / y);
    const MhRecip r = mh_denom(y);
    bool bad = r.bad;
    const double q = mh_div(x, r, bad);
    if (!bad) div += !equal(q, x / y);
    lim += !gradient<0>(x, y) + !gradient<1>(x, y) + !gradient<2>(x, y) + !gradient<3>(x, y);
    ++pairs;
  }
  std::printf("%ld %ld %ld\n", pairs, div, lim);
  return 0;
}
