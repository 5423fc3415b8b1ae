// Host check of GenTile (mh_geom.h): for meshes nx nt na on stdin, prints the cells that no thread or
// more than one updates, the updated cells whose face ahead is not the next row's, and the threads launched.
#include <cstdio>
#include <vector>
#include "../../mahyco_amd/csrc/mh_geom.h"

int main() {
  int nx, nt, na;
  while (std::scanf("%d %d %d", &nx, &nt, &na) == 3) {
    const GenTile tile(nx, nt, na);
    std::vector<int> seen((size_t)nx * nt * na, 0);
    long ahead = 0;
    const long blocks = (tile.blocks() + 7) / 8 * 8;  // as launched
    for (long lb = 0; lb < blocks; ++lb)
      for (int tid = 0; tid < 256; ++tid) {
        int i, t, a;
        if (!tile.face((int)lb, tid, i, t, a) || !tile.cell(tid)) continue;
        if (i < 0 || i >= nx || t < 0 || t >= nt || a < 0 || a >= na) return 1;
        ++seen[i + (size_t)nx * (t + (size_t)nt * a)];
        if (a + 1 < na) {
          int i2, t2, a2;
          ahead += tid + (1 << tile.lx) >= 256 || !tile.face((int)lb, tid + (1 << tile.lx), i2, t2, a2) || i2 != i || t2 != t || a2 != a + 1;
        }
      }
    long bad = 0;
    for (int s : seen) bad += s != 1;
    std::printf("%ld %ld %ld\n", bad, ahead, blocks * 256);
  }
  return 0;
}
