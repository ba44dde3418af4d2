// Which of the kernels of sgemm_split.hip takes an fp32 product, if any.  A plain function of integers, compiled for the
// dispatcher and for the tests, which ask it for the route of each of their shapes.
#pragma once

#include "sgemm_tiles.hpp"

namespace tfcc_rocm {
namespace sgemm_split_plan {

enum Kernel { kNone = -1, kWide = 0, k128 = 1, k64 = 2 };  // tiles of 128 x 256, 128 x 128, 64 x 64 with four K groups

// K groups of 128 x 128 tiles: two, as eight wavefronts of one workgroup, while a CU has one tile at most.  A wavefront for
// each SIMD waits for its slabs, and nothing of another one's runs meanwhile: us with one and with two, 2048^3 101 -> 92, 1024 x
// 768 x 3072 40 -> 35, 328 x 1536 x 4678 64 -> 53; of 546 products 0.95 of the time up to 200 k, 0.89 around 350 and 0.82 from 900
// on, but more than that with many tiles of a short K, which the meeting of the groups makes longer.  (With two tiles for a CU
// their workgroups run side by side: 2304 x 3584 x 3200 256, and 255 with two groups.)
inline int k_groups_of_128(unsigned long long tiles, unsigned depth) { return tiles <= 256 && (depth >= 320 || tiles <= 128) ? 2 : 1; }

// Measured times, from 64 to 1536 tiles of 128 x 128 and K from 192 to 4096, are met within a fifth by a constant, one per
// round of tiles, and K times what a CU takes for a k with one, two, ... tiles on it (as soon as one CU has two 128 x 128
// tiles all of it takes three quarters of what it takes when all have two; 64 x 64 tiles are multiple); the kernels on the
// fp32 matrix ops reach some 115 TFLOP/s, 105 where a K or an N is no multiple of their pieces, and more on large products,
// which have the most to gain here.  Of 420 shapes, even over the logarithm of 64 .. 4096 rows and 64 .. 8192 for K and N, up to
// 2^35 products, 60 come here, 1.43 times as fast on the average and none slower; 150 others that come here take 0.70 of their
// time, one of them 1.02 (4096^3: 910 -> 602 us, to 641 by the card).  The larger tiles take
// what they are thought to be faster at: 38 shapes within a tenth of that line take 1.0 to 1.9 times as long on the fp32 ops up
// to it, and 0.98 to 1.5 times from it on.  64 x 64 tiles have to be faster by an eighth, and by a quarter where the product
// takes less than 60 us otherwise: those that are not gain 6 % on the average and lose up to 7 (704 x 2847 x 455), and in a layer
// of other products less than nothing, because these run a microsecond or two longer behind them.  128 x 128 tiles with two
// K groups, which have to be faster by an eighth, are worth it there: a served layer of 8 x 128 x 768 294 -> 286.
// A true batch of short products keeps the kernels whose sums the attention kernel reproduces.
inline int kernel_of(unsigned rows, unsigned columns, unsigned depth, unsigned lda, unsigned ldb, unsigned ldc, bool transB, unsigned batch) {
  const unsigned long long m = rows, n = columns, k = depth;
  if (m < 48 || n < 48 || k < (batch > 1 ? 192u : 128u)) return kNone;
  // byte offsets of whole operands and of a tile's rows of the result fit 31 and 30 bits
  if ((m + 256) * lda >= (1u << 29) || ((transB ? n : k) + 256) * ldb >= (1u << 29) || ldc >= (1u << 21)) return kNone;
  auto tiles = [&](unsigned rowsOf, unsigned columnsOf) { return ((m + rowsOf - 1) / rowsOf) * ((n + columnsOf - 1) / columnsOf) * batch; };
  const unsigned long long t64 = tiles(64, 64), t128 = tiles(128, 128), wide = tiles(128, 256);
  if (t64 < 128) return kNone;
  auto costWide = [&] {
    const unsigned long long full = wide / 256, r = wide % 256;
    return 8 + 3.2 * (full + (r != 0)) + k * (full * .0743 + (r ? .048 + r * r * 4e-7 : 0));
  };
  // What the fp32 ops take, by operations and by tiles: the larger one, for what leaves CUs without work there is what there is
  // to gain here (328 x 1536 x 4678: 64 us, 49 by operations, 41 in 128 x 128 tiles).  Of 120000 drawn products 9000 go another way than
  // by operations and with one K group alone.  6600 of those, timed: 0.80 of the time in cache, 0.82 from memory; 17 take more than
  // 1.03 in cache, most in batches of 64 to 82 rows (64 x 268 x 7872, 32 of them, 1.11; 75 x 7958 x 558, 40, 1.13), and 410 from memory, nearly
  // all single products that leave 64 x 64 tiles for two K groups: these take 0.92 in cache and 1.00 from memory, 1.17 at most
  // (2752 x 5539 x 896).  Where the fp32 ops have 128 x 128 tiles as well, operations alone decide: that estimate is nearer there.
  const double rate = k % 32 != 0 || n % 4 != 0 ? 105e6 : 115e6;  // operations in a microsecond
  const double byTiles = sgemm_tiles::microseconds(rows, columns, depth, batch), byOperations = 4 + 2. * m * n * k * batch / rate;
  const double below = byTiles > byOperations ? byTiles : byOperations;
  const bool twice = byTiles != 0 && k_groups_of_128(t128, depth) == 2;
  auto cost128 = [&] {
    if (twice) return 8.5 + k * (.0265 + (t128 > 90 ? (t128 - 90) * .00007 : 0));
    const unsigned long long r = t128 % 512;
    return 9 + k * (t128 / 512 * .0813 + (r == 0 ? 0 : r <= 256 ? .0403 : .06 + (r - 256) * .00008));
  };
  auto cost64 = [&] { return 4 + 4.5 * ((t64 + 511) / 512) + k * .0108 * ((t64 + 255) / 256); };
  const double costs[3] = {costWide(), cost128(), cost64()};
  int best = costs[0] <= costs[1] && costs[0] <= costs[2] ? kWide : costs[1] <= costs[2] ? k128 : k64;
  const double margin64 = below < 60 ? .75 : .87;
  // A batch whose operands nothing reads twice comes from memory, and then a long K takes two K groups longer than that, rows at odd
  // addresses most (1956 x 2559 x 112, 12 of them, 139 us, 105 estimated and 109 in 64 x 64 tiles).  209 products that have 64 x 64 tiles
  // for it took 0.97 of their time in the others in cache, 1.02 from memory, 33 more than 1.03 in both, up to 1.27.
  if (batch > 1 && twice && best == k128 && k >= 2500 && costs[k64] < margin64 * byOperations &&
      costs[k64] < (k % 4 == 0 ? 1.08 : 1.2) * costs[k128])
    best = k64;
  const double margin = best == k64 ? margin64 : best == k128 && twice ? .88 : 1.;
  // One K group, but so many k that the fp32 ops have two: up to 1.03 of their time in cache and 1.12 from memory (704 x 312 x
  // 3656) where it is thought to be no faster than by a tenth.
  const double marginByTiles = best == k128 && !twice && k >= 300 ? .9 : .92;
  return costs[best] < margin * byOperations || costs[best] < (margin < marginByTiles ? margin : marginByTiles) * byTiles ? best : kNone;
}

}  // namespace sgemm_split_plan
}  // namespace tfcc_rocm
