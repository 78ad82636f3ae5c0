// Rows of a leaf's AO planes that a column block's wavefronts read
// (occ_amd/csrc/tile_shapes.hpp), for every number of AOs a leaf may have and
// every block width: a wavefront reads 16 rows a tile of its half block from the
// half's first row on, which must stay below the padded row count, and the tiles
// of all halves must hold every real AO once.  Exit status 1 if any fails.
#include <cstdio>

#include "tile_shapes.hpp"

using namespace occxc;

int main() {
  int failed = 0;
  for (int maxw = 32; maxw <= 128; maxw += 32)
    for (int m = 1; m <= 8192; ++m) {
      const int mp = (m + 31) / 32 * 32;
      int next = 0, largest = -1, real = 0;
      bool ok = true;
      for (const auto &b : tile_blocks(mp, maxw)) {
        ok = ok && b.first == next && b.second >= 32 && b.second <= maxw;
        next += b.second;
        for (int half = 0; half < 2; ++half) {
          const int hc = b.second / 2, row0 = b.first + half * hc;
          const int tiles = half_tiles(m - row0, hc);
          ok = ok && hc % 16 == 0 && 16 * tiles <= hc;  // no row of the other half
          for (int r = row0; r < row0 + 16 * tiles; ++r) real += r < m;
          if (tiles > 0 && row0 + 16 * tiles - 1 > largest) largest = row0 + 16 * tiles - 1;
        }
      }
      if (ok && next == mp && largest < mp && real == m) continue;
      if (++failed <= 10)
        std::printf("blocks of %d: %d AOs, %d rows, row %d read\n", maxw, m, mp, largest);
    }
  std::printf("%d failed checks\n", failed);
  return failed != 0;
}
