// Size and order of the GEMM's output tiles (no HIP headers: the tests compile this file by
// itself, with cdiv and GEMM_BK).
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

// Estimated time (us) of `tiles` workgroups, `per_cu` of them resident on a CU, over ns
// 128-byte stages of K: a start-up cost, then per round t1 per stage with one workgroup on a
// CU or t2 with two, and the LoRA branch's `lora` per workgroup on a CU.
inline float gemm_time(int64_t tiles, int cus, int per_cu, int64_t ns, float start, float t1, float t2, float lora) {
  if (per_cu == 1) return start + (float)cdiv(tiles, cus) * (t1 * (float)ns + lora);
  const int64_t full = tiles / (2 * cus), rem = tiles - full * 2 * cus;
  return start + (float)full * (t2 * (float)ns + 2.0f * lora) +
         (rem == 0 ? 0.0f : rem <= cus ? t1 * (float)ns + lora : t2 * (float)ns + 2.0f * lora);
}

// The tile of an M x N x K product with a LoRA of rank r (0 without): 0-3 a ring tile, 32 x 64,
// 64 x 64, 128 x 64 or 128 x 128 (gemm_ring.h), else 128 x 128 or 256 x 256 tiles of
// gemm_fp8_rowwise_kernel.
//
// 256 x 256 tiles from 512 of them on, always.  Below that the fastest by these estimates,
// where another tile replaces the 128 x 128 ones only if it saves a twentieth, and the
// 256 x 256 ones only where they make one round over the CUs (two rounds gained with cold weights
// and lost with warm ones: 2048 x 9216 x 3072 87 -> 73 and 63 -> 72 us).
//
// The constants are fitted to MI355X times (graph replays; weights from HBM with warm
// activations, and both warm) of 680 products without a LoRA (M 1-20000, N 64-12288, K 512-12288)
// and 660 with ranks of 16 to 4096.  Over those, with cold / warm weights, the choice took
// 0.80 / 0.83 of the time of 128 x 128 tiles (256 x 256 from 512) without a LoRA, 0.75 / 0.80
// up to rank 128 and 0.65 / 0.67 above, 1-2% longer than the best tile each time.  At worst it took
// 1.03 of their time without a LoRA (1.10 with everything warm: 14296 x 256 x 1024 9.2 against
// 8.3 us), 1.00 up to rank 128 and 1.06 above.
// What the terms stand for: the ring tiles gain most where M leaves CUs without a 128 x 128
// tile (1 x 3072 x 3072 17.0 -> 8.2 us, 1024 x 3072 x 12288 105 -> 66); past that the larger
// tile reads fewer operand bytes (2048 x 3072 x 3072 23.8 us against 28.0 with 128 x 64), and
// where nearly every slot has a tile their deep rings start slower (`full`).  A LoRA is read from
// LDS up to rank 128 and from global memory above by the two kernels of 128 x 128 and 256 x 256
// tiles; the latter, one workgroup per CU, then waits most (2048 x 3072 x 3072 at rank 1024:
// 253 us, 131 with 128 x 128, 112 with ring tiles of 128 x 64).
enum { GEMM_TILE_128 = 4, GEMM_TILE_256 = 5 };
inline int gemm_pick(int64_t M, int64_t N, int64_t K, int64_t r, int cus) {
  const int64_t ns = cdiv(K, GEMM_BK);
  const float l = (float)r / 64.0f, saves = 0.95f;
  auto tiles = [&](int bm, int bn) { return cdiv(M, bm) * cdiv(N, bn); };
  const int64_t big_tiles = tiles(256, 256);
  if (big_tiles >= 2 * 256) return GEMM_TILE_256;
  const int64_t t64 = tiles(128, 64), t128 = tiles(128, 128);
  auto full = [](int64_t t, int slots) { return t <= slots && t > slots * 7 / 8 ? 0.5f : 0.0f; };
  float time = gemm_time(t128, cus, 2, ns, 4.4f, 0.68f, 0.87f, (r <= 128 ? 1.0f : 3.2f) * l);
  const float ring[4] = {gemm_time(tiles(32, 64), cus, 1, ns, 2.8f, 0.24f, 0.0f, 0.7f * l),
                         gemm_time(tiles(64, 64), cus, 2, ns, 4.0f, 0.28f, 0.465f, 1.0f * l),
                         gemm_time(t64, cus, 2, ns, 4.0f + full(t64, 2 * cus), 0.315f, 0.615f, 1.5f * l),
                         gemm_time(t128, cus, 1, ns, 4.6f + full(t128, cus), 0.54f, 0.0f, 3.4f * l)};
  int best = 0;
  for (int i = 1; i < 4; ++i)
    if (ring[i] < ring[best]) best = i;
  int pick = GEMM_TILE_128;
  if (ring[best] <= saves * time) pick = best, time = ring[best];
  if (big_tiles <= cus &&
      gemm_time(big_tiles, cus, 1, ns, 6.4f, 1.16f, 0.0f, (r <= 128 ? 2.6f : 11.0f) * l) <= saves * time)
    pick = GEMM_TILE_256;
  return pick;
}

}  // namespace mxf8
