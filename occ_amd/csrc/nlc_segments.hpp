// nlc_segments.hpp -- how the VV10 pair sum is cut into units of work: the one
// place that the kernel which writes the partial sums, the kernel which adds
// them up and the size of their buffer take it from.  Plain C++, so that a host
// test can compare the three over every number of points.
#pragma once

namespace occxc {

constexpr int kVvTile = 256;   // j points of a tile
constexpr int kVvRows = 512;   // i points of a block, two per thread
constexpr int kVvSegs = 16;    // most segments of j

constexpr long long vv_tiles(long long npts) { return (npts + kVvTile - 1) / kVvTile; }
constexpr long long vv_blocks(long long npts) { return (npts + kVvRows - 1) / kVvRows; }

// Segments of j: runs of `tiles` tiles, so that the triangle of pairs becomes
// many units of about equal work (one workgroup per 256 points with all of its
// j tiles left a quarter of the chip idle at the end: 1032 workgroups, all
// resident at once, the longest twice the average).
struct VvSegs {
  int tiles, n;
};
constexpr VvSegs vv_segs(long long npts) {
  const long long nt = vv_tiles(npts), per = (nt + kVvSegs - 1) / kVvSegs;
  const long long tiles = per < 8 ? 8 : per, n = (nt + tiles - 1) / tiles;
  return VvSegs{(int)tiles, (int)(n < 1 ? 1 : n)};
}

// Block b's j tiles are 0 .. vv_last_tile: up to its own two, of which the
// second does not exist where the number of tiles is odd and b is the last.
constexpr long long vv_last_tile(long long b, long long npts) {
  return 2 * b + 1 < vv_tiles(npts) ? 2 * b + 1 : vv_tiles(npts) - 1;
}
// the segments 0 .. vv_block_segs - 1 hold them
constexpr int vv_block_segs(long long b, long long npts, int seg_tiles) {
  return (int)(vv_last_tile(b, npts) / seg_tiles) + 1;
}

} // namespace occxc
