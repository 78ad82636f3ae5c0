// The units that the VV10 pair sum is cut into (occ_amd/csrc/nlc_segments.hpp),
// for every number of points up to 5e5 (1954 tiles, two point counts of each)
// and some larger ones: each block's j tiles, 0 up to its own last one and none
// past the points, are walked exactly once by the launched segments, and the
// segments that the sums add up are the written ones and lie in the buffer.
// Exit status 1 if any fails.
#include <cstdio>
#include <initializer_list>

#include "nlc_segments.hpp"

using namespace occxc;

static bool covered(long long npts) {
  const VvSegs g = vv_segs(npts);
  const long long nt = (npts + kVvTile - 1) / kVvTile;
  for (long long b = 0; b < vv_blocks(npts); ++b) {
    const int read = vv_block_segs(b, npts, g.tiles);
    if (read < 1 || read > g.n) return false;  // launched, and in the buffer
    // the tiles that hold points at or before the block's last point
    const long long last_i = (b + 1) * kVvRows < npts ? (b + 1) * kVvRows - 1 : npts - 1;
    const long long need = last_i / kVvTile;
    long long next = 0;
    for (int seg = 0; seg < read; ++seg) {
      const long long j0 = (long long)seg * g.tiles, end = vv_last_tile(b, npts) + 1;
      const long long j1 = j0 + g.tiles < end ? j0 + g.tiles : end;
      if (j0 != next || j1 <= j0 || j1 > nt) return false;
      next = j1;
    }
    if (next != need + 1) return false;
  }
  return true;
}

int main() {
  int failed = 0;
  auto check = [&](long long npts) {
    if (covered(npts)) return;
    ++failed;
    std::printf("npts %lld: segments %d of %d tiles\n", npts, vv_segs(npts).n, vv_segs(npts).tiles);
  };
  for (long long nt = 1; nt <= 1954; ++nt)
    for (long long npts : {(nt - 1) * kVvTile + 1, nt * kVvTile}) check(npts);
  for (long long npts : {1000000LL, 1048577LL, 3999999LL, 8697600LL}) check(npts);
  std::printf("%d failed checks\n", failed);
  return failed != 0;
}
