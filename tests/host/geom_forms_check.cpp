// Host check of the scaled corner-vector forms in mh_geom.h: cqs_hex_each, cqs_hex_corner<L> and
// hex_volume must give the bits of cqs_hex and cell_volume<8>.  Reads hexahedra (24 doubles each,
// as hexadecimal bit patterns) on stdin, prints the cells read and the number of mismatches.
#include <cinttypes>
#include <cstdio>
#include <cstring>
#include "../../mahyco_amd/csrc/mh_geom.h"

static uint64_t bits(double v) { uint64_t u; std::memcpy(&u, &v, 8); return u; }
static double from_bits(uint64_t u) { double v; std::memcpy(&v, &u, 8); return v; }
static bool same(const D3& a, const D3& b) {
  return bits(a.x) == bits(b.x) && bits(a.y) == bits(b.y) && bits(a.z) == bits(b.z);
}

int main() {
  long cells = 0, bad = 0;
  for (;;) {
    uint64_t raw[24];
    int got = 0;
    for (int k = 0; k < 24; ++k) got += std::scanf("%" SCNx64, &raw[k]);
    if (got != 24) break;
    D3 x[8], q[8], e[8];
    for (int l = 0; l < 8; ++l) x[l] = d3(from_bits(raw[3 * l]), from_bits(raw[3 * l + 1]), from_bits(raw[3 * l + 2]));
    cqs_hex(x, q);
    cqs_hex_each(x, [&](int l, const D3& v) { e[l] = v; });
    const D3 c[8] = {cqs_hex_corner<0>(x), cqs_hex_corner<1>(x), cqs_hex_corner<2>(x), cqs_hex_corner<3>(x),
                     cqs_hex_corner<4>(x), cqs_hex_corner<5>(x), cqs_hex_corner<6>(x), cqs_hex_corner<7>(x)};
    for (int l = 0; l < 8; ++l) bad += !same(q[l], e[l]) + !same(q[l], c[l]);
    bad += bits(hex_volume(x)) != bits(cell_volume<8>(x, q, 3));
    ++cells;
  }
  std::printf("%ld %ld\n", cells, bad);
  return 0;
}
