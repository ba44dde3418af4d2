// Which of the kernels of sgemm_split.hip takes an fp32 product, if any.  A plain function of integers, compiled for the
// dispatcher and for the tests, which ask it for the route of each of their shapes.
#pragma once

namespace tfcc_rocm {
namespace sgemm_split_plan {

enum Kernel { kNone = -1, kWide = 0, k128 = 1, k64 = 2 };  // tiles of 128 x 256, 128 x 128, 64 x 64 with four K groups

// Measured times, from 64 to 1536 tiles of 128 x 128 and K from 192 to 4096, are met within a fifth by a constant, one per
// round of tiles, and K times what a CU takes for a k with one, two, ... tiles on it (as soon as one CU has two 128 x 128
// tiles all of it takes three quarters of what it takes when all have two; 64 x 64 tiles are multiple); the kernels on the
// fp32 matrix ops reach some 115 TFLOP/s, 105 where a K or an N is no multiple of their pieces, and more on large products,
// which have the most to gain here.  Of 420 shapes, even over the logarithm of 64 .. 4096 rows and 64 .. 8192 for K and N, up to
// 2^35 products, 60 come here, 1.43 times as fast on the average and none slower; 150 others that come here take 0.70 of their
// time, one of them 1.02 (4096^3: 910 -> 602 us, to 641 by the card).  The larger tiles take
// what they are thought to be faster at: 38 shapes within a tenth of that line take 1.0 to 1.9 times as long on the fp32 ops up
// to it, and 0.98 to 1.5 times from it on.  64 x 64 tiles have to be
// faster by an eighth, and by a quarter where the product takes less than 60 us otherwise: those that are not gain 6 % on the average and lose up to
// 7 (704 x 2847 x 455), and in a layer of other products less than nothing, because these run a microsecond or two longer
// behind them (1024 x 768 x 3072 with GELU 38.7 us here and 41.8 on the fp32 ops, the layer around it 326 and 320).
// A true batch of short products keeps the kernels
// whose sums the attention kernel reproduces.
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
  auto cost128 = [&] {
    const unsigned long long r = t128 % 512;
    return 9 + k * (t128 / 512 * .0813 + (r == 0 ? 0 : r <= 256 ? .0403 : .06 + (r - 256) * .00008));
  };
  auto cost64 = [&] { return 4 + 4.5 * ((t64 + 511) / 512) + k * .0108 * ((t64 + 255) / 256); };
  const double costs[3] = {costWide(), cost128(), cost64()};
  const int best = costs[0] <= costs[1] && costs[0] <= costs[2] ? kWide : costs[1] <= costs[2] ? k128 : k64;
  const double rate = k % 32 != 0 || n % 4 != 0 ? 105e6 : 115e6;  // operations in a microsecond
  const double below = 4 + 2. * m * n * k * batch / rate;
  return costs[best] < (best != k64 ? 1. : below < 60 ? .75 : .87) * below ? best : kNone;
}

}  // namespace sgemm_split_plan
}  // namespace tfcc_rocm
