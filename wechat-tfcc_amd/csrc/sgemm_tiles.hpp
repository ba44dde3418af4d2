// Which tiles an fp32 product takes on the fp32 matrix ops, and about how long that is.  Plain functions of integers, compiled
// for the dispatcher and, with the rule of sgemm_split_plan.hpp, for the tests.
#pragma once

namespace tfcc_rocm {
namespace sgemm_tiles {

// The tile table of the kernels that copy K slabs straight into LDS, ordered by falling tile area.
constexpr struct { int config; unsigned bm, bn, waves; } kTiles[] = {{0, 64, 64, 4}, {1, 32, 96, 3}, {2, 32, 64, 2}, {3, 32, 32, 1}};

inline unsigned long long tiles_of(unsigned m, unsigned n, unsigned batch, unsigned bm, unsigned bn) {
  return (unsigned long long)((m + bm - 1) / bm) * ((n + bn - 1) / bn) * batch;
}

// Tile and number of K groups for m x n x k with K a multiple of 32: the tile that covers the 256 CUs in the fewest
// tile-area rounds, the larger one on a tie (less operand traffic); as few K groups as give every CU eight
// wavefronts, each group keeping at least four slabs.
inline void choose_dma_tiles(unsigned m, unsigned n, unsigned k, unsigned fillBatch, int& best, unsigned long long& bestTiles,
                             int& ksplit) {
  best = 0;
  unsigned long long bestCost = ~0ull;
  bestTiles = 0;
  for (int c = 0; c < 4; ++c) {
    const unsigned long long tiles = tiles_of(m, n, fillBatch, kTiles[c].bm, kTiles[c].bn);
    const unsigned long long cost = ((tiles + 255) / 256) * (kTiles[c].bm * kTiles[c].bn);
    if (cost < bestCost) {
      best = c;
      bestCost = cost;
      bestTiles = tiles;
    }
  }
  ksplit = 1;
  while (ksplit < 4 && bestTiles * kTiles[best].waves * ksplit < 256ull * 8 && k >= 128u * (ksplit * 2)) ksplit *= 2;
}

// 128 x 128 tiles: once there are enough of them to fill the 256 CUs twice over, and only when they are mostly
// result (a batch of 768 products of 64 x 64 x 64 counts 768 such tiles, each three quarters empty: 23 us in them
// against 11 in 64 x 64 tiles).
inline bool takes_128_tiles(unsigned m, unsigned n, unsigned fillBatch) {
  const unsigned long long big = tiles_of(m, n, fillBatch, 128, 128);
  return big >= 512 && (unsigned long long)m * n * fillBatch * 100 >= big * (128 * 128) * 75;
}

// Without K groups: the products whose 128 x 96 tiles fill at least 70 % of the CUs in each of their rounds (or 128 x 128
// tiles 85 %), K >= 512: four wavefronts of 32 x 96 (32 x 128) share each copy of B (1024 x 3072 x 768 with GELU: 39.3 against
// 42.4 us in 64 x 64 tiles, 1536^3: 69 against 80; below those fills, or with a short K, the table's win).  3 or 4 blocks of 32
// columns, or 0.
inline int shared_blocks(unsigned m, unsigned n, unsigned k, unsigned fillBatch, int ksplit) {
  if (ksplit != 1 || k < 512) return 0;
  const unsigned long long wide = tiles_of(m, n, fillBatch, 128, 96), wide4 = tiles_of(m, n, fillBatch, 128, 128);
  const bool ok3 = wide * 100 >= 70 * 256 * ((wide + 255) / 256), ok4 = wide4 * 100 >= 85 * 256 * ((wide4 + 255) / 256);
  const unsigned long long cost3 = ((wide + 255) / 256) * 96, cost4 = ((wide4 + 255) / 256) * 128;
  return ok4 && (!ok3 || cost4 < cost3) ? 4 : ok3 ? 3 : 0;
}

// Microseconds that the product takes, or 0 where it has 128 x 128 tiles: a constant, and for the area that the busiest CU
// has to do, in tiles of 64 x 64, something per k and once.  Fitted to 860 products of 64 to 4096 rows, K and N from 64 to 8192;
// met within 6 % on the average, a fifth at most.
inline double microseconds(unsigned m, unsigned n, unsigned k, unsigned fillBatch) {
  if (takes_128_tiles(m, n, fillBatch)) return 0;
  constexpr struct { double base, perK, once; } kTimes[4][3] = {  // one, two and four K groups
      {{3.4, .0158, .7}, {2.7, .0149, 1.2}, {2.0, .0153, 2.0}},   // 64 x 64
      {{4.0, .0221, .6}, {3.9, .0216, 1.4}, {2.7, .0146, 2.0}},   // 32 x 96
      {{4.5, .0225, .6}, {3.5, .0170, 1.5}, {1.0, .0155, 4.4}},   // 32 x 64
      {{4.0, .0251, .3}, {3.4, .0212, -.6}, {1.0, .0237, 1.1}}};  // 32 x 32
  int best, ksplit;
  unsigned long long tiles;
  choose_dma_tiles(m, n, k, fillBatch, best, tiles, ksplit);
  const int shared = shared_blocks(m, n, k, fillBatch, ksplit);
  if (shared == 4) return 0;
  auto time = [&](unsigned long long count, unsigned area, double base, double perK, double once) {
    return base + (k * perK + once) * ((count + 255) / 256 * area) / 4096;
  };
  if (shared == 3) return time(tiles_of(m, n, fillBatch, 128, 96), 128 * 96, 6.1, .0141, .2);
  const auto& t = kTimes[best][ksplit >> 1];
  return time(tiles, kTiles[best].bm * kTiles[best].bn, t.base, t.perK, t.once);
}

}  // namespace sgemm_tiles
}  // namespace tfcc_rocm
