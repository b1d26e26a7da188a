// Order of the GEMM's output tiles (no HIP headers: the tests compile this file by itself).
#pragma once

namespace mxf8 {

// Map a tile sequence number s to an output tile.  Workgroups are dealt to the 8 XCDs
// round-robin and a persistent workgroup b walks s = b, b + G, b + 2G, ... (G = grid, a
// multiple of 8), so s % 8 names the XCD: give every XCD a contiguous range of tile ids,
// then walk that range in groups of group_m token-tiles so concurrently running tiles
// share operand panels in the XCD's L2.
__host__ __device__ inline void tile_coords(int s, int tiles_m, int tiles_n, int group_m, int& tm, int& tn) {
  const int nwg = tiles_m * tiles_n;
  const int q = nwg >> 3, rem = nwg & 7, x = s & 7, j = s >> 3;
  const int id = (x < rem ? x * (q + 1) : rem * (q + 1) + (x - rem) * q) + j;
  const int per_group = group_m * tiles_n;
  const int g = id / per_group;
  const int first_m = g * group_m;
  const int gsize = min(tiles_m - first_m, group_m);
  const int in = id - g * per_group;
  tm = first_m + in % gsize;
  tn = in / gsize;
}

// Token-tiles per group of the short-token kernel (gemm_ring.h), one tile per workgroup.  Up to
// 8 token-tiles are one group: the tiles that share a weight panel, which comes from HBM, run on
// one XCD.  More tokens than that would fill an XCD with the tiles of one or two weight panels,
// each with an activation panel of its own, and every activation panel would be read by each
// channel tile's XCD.  MI355X, all token-tiles in one group -> groups of 8: 19160 x 192 x 4096
// 35.8 -> 24.0 us, 16344 x 256 x 6144 35.0 -> 31.4, 4056 x 1024 x 2048 16.5 -> 14.0,
// 6144 x 640 x 3072 20.6 -> 18.3 us (groups of 4 within 5% of these, of 16 up to 9% slower).
constexpr int RING_GROUP_M = 8;

}  // namespace mxf8
