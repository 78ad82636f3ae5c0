// tile_shapes.hpp -- how a leaf's AOs are cut into blocks and a block's halves
// into 16-row MFMA tiles.  Plain C++ (constexpr functions serve kernels too), so
// that a host test can check the rows that a kernel reads.
#pragma once

#include <utility>
#include <vector>

namespace occxc {

// 16-row tiles of a wavefront's half block (half rows, a multiple of 16) that
// hold any of the `valid` rows counted from its first row.  The tiles past a
// leaf's real AOs or points hold padding only (zero AO rows, zero-weight
// points).
constexpr int half_tiles(int valid, int half) {
  return ((valid < 0 ? 0 : valid < half ? valid : half) + 15) >> 4;
}

// Blocks of a leaf's padded AOs: n / 32 units of 32 split into the fewest
// blocks of at most maxw / 32 units, the first ones one unit larger.
inline std::vector<std::pair<int, int>> tile_blocks(int n, int maxw) {
  std::vector<std::pair<int, int>> b;
  const int per = maxw < 32 ? 1 : maxw / 32;
  const int units = n / 32, nb = (units + per - 1) / per;
  int at = 0;
  for (int k = 0; k < nb; ++k) {
    const int u = units / nb + (k < units % nb ? 1 : 0);
    b.push_back({at, 32 * u});
    at += 32 * u;
  }
  return b;
}

} // namespace occxc
