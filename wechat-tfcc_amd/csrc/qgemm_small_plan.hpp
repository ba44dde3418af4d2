// How a small quantized product is dealt out over workgroups (gemm_u8s8_small.hip).  A plain function of integers, compiled for
// the launcher and for the tests, which ask it for the route of their shapes.
#pragma once

namespace tfcc_rocm {
namespace qgemm_small_plan {

// Rows per tile and wavefronts by the amount of work, in steps of 16 rows x 64 columns x 64 k (measured, us):
//   up to 4096 steps, or at most 16 rows, tiles of 16 rows: there latency is all there is, and the most workgroups share
//     it (77 x 1001 x 1237: 7.1 in 16 rows, 8.2 in 32, 11.3 in 64);
//   from there tiles of 32 rows, which load half as much of B per product (128 x 768 x 3072: 6.3 against 6.9);
//   above 12000 steps tiles of 64 rows while there are 128 of them (700 x 2001 x 803: 18.6 against 21.2 and 22.7; 100 x
//     4001 x 4003, 126 tiles: 34 against 22 in 32 rows).
// Wavefronts: 4 for at most six steps of k, or when 8 of each tile would be more than eight per CU (1024 x 768 x 768 in 32
// rows: 8.1 with 4, 10.8 with 8); 16 on the smallest tiles when they are few and K is long (32 x 3292 x 704: 8.4 against
// 8.7 and 10.7 with 8 and 4); 8 otherwise.
//
// A tile's steps go to several workgroups, in tiles of 16 rows, where that saves more trips to memory than the meeting costs.
// Microseconds as first measured: a pair of steps of every worker is a trip, and a launch takes 3.0 + 1.2 for each trip of
// four wavefronts, 3.8 + 1.8 of eight, 4.2 + 3 of sixteen, 4 + 2.1 (1.7) in 32 rows of eight (four); the meeting takes 2.4 as
// long as there are at most eight wavefronts on a CU.  These choose the number of workgroups: 0.7 is asked for on top, and
// more than 20 steps (with the operands in cache 8 x 920 x 552 takes 6.1 in one piece and 6.5 in three).
// Whether they are better than one was then fitted to 600 products that these rules split, drawn evenly over the logarithm of
// 1 .. 2048 rows, 800 .. 12288 for K and 16 .. 8192 for N, each with its operands in cache: time depends on the steps, on
// rows of A and of B that begin at odd addresses, and on the wavefronts for each CU.  The fit refuses 49 of the 600,
// which took 1.14 times as long split with the operands in cache and 1.03 from HBM.  Of 500 others, drawn the same way, that
// the two rules looked at, none is slower than in one piece from HBM and three are from the cache, by up to 1.12; on the
// average they take 0.58 and 0.63 of the time.  3 x 11304 x 910 27.3 -> 9.3, 32 x 8192 x 512 18.5 -> 7.8, 99 x 3481 x 512
// 11.7 -> 7.8; 526 x 1832 x 400 stays at 7.5 (10.2 split).
// Where up to three trips would take more wavefronts than that, four to eight do: of 60 such products, one in twelve of those of
// more than 1300 k that come here, the 40 that are thought to take three quarters of the time at most take 0.72 of it, none more than 0.98
// (43 x 7005 x 1920 25.5 -> 12.1, 830 x 5881 x 96 22.8 -> 11.3, 29 x 7565 x 4331 35.5 -> 21.4); the others 0.98, up to 1.12 (221 x 4120 x 1101
// 15.9 -> 17.8).
constexpr int kCols = 64;                   // columns of a tile
constexpr unsigned kMaxResults = 1u << 19;  // of a product that is split

struct Plan {
  unsigned rows, waves;         // of a workgroup that has all of K
  unsigned splits, splitWaves;  // of tiles of 16 rows; splits 1: not better
  unsigned cost, splitCost;     // hundredths of a microsecond
  bool better;                  // split, than in one piece
};
inline Plan plan_of(unsigned m, unsigned n, unsigned k, unsigned batch) {
  const unsigned steps = (k + 63) / 64;
  const unsigned long long columns = (unsigned long long)((n + 63) / 64) * batch;
  const unsigned long long tiles16 = (m + 15) / 16 * columns, tiles32 = (m + 31) / 32 * columns, tiles64 = (m + 63) / 64 * columns;
  const unsigned long long work = tiles16 * steps;
  Plan p{16, 8, 1, 0, 0, ~0u, false};
  if (work > 12000 && tiles64 >= 128) p.rows = 64, p.waves = steps <= 6 ? 4 : 8;
  else if (work > 4096 && m > 16) p.rows = 32, p.waves = steps <= 6 || tiles32 * 8 > 2048 ? 4 : 8;
  else if (steps <= 6 || tiles16 * 8 > 2048) p.waves = 4;
  else if (tiles16 <= 128 && steps >= 30) p.waves = 16;
  auto trips = [&](unsigned waves) { return (steps + 2 * (waves - 1) - 1) / (2 * (waves - 1)); };
  p.cost = p.rows == 32 ? 400 + (p.waves == 4 ? 170 : 210) * trips(p.waves)
                        : p.waves == 4 ? 300 + 120 * trips(4) : p.waves == 8 ? 380 + 180 * trips(8) : 420 + 300 * trips(16);
  if (steps <= 20 || p.rows == 64 || tiles16 * 16 * kCols > kMaxResults) return p;
  auto choose = [&](unsigned waves, unsigned least, unsigned most, double margin) {
    for (unsigned want = least; want <= most; ++want) {  // trips
      const unsigned splits = (steps + 2 * (waves - 1) * want - 1) / (2 * (waves - 1) * want);
      const unsigned cost = (waves == 4 ? 300 + 120 * want : 380 + 180 * want) + 240;
      if (splits < 2 || splits > 32 || tiles16 * splits * waves > 2048 || cost + 70 > p.cost || cost >= p.splitCost) continue;
      p.splits = splits;
      p.splitWaves = waves;
      p.splitCost = cost;
      const double oddA = k % 4 != 0, oddB = n % 4 != 0, odd = oddA + oddB;
      const double tiles = p.rows == 32 ? tiles32 : tiles16, all = tiles * p.waves / 256, shared = tiles16 * splits * waves / 256.;
      const double one = p.rows == 32    ? 240 + steps * (10.5 + 9 * oddA + 4 * oddB) + all * (3. * steps - 10)
                         : p.waves == 16 ? 490 + steps * (5.6 + 3.8 * oddA + 3.6 * oddB) + all * (3.1 * steps - 91)
                                         : 600 + steps * 3.5 * odd + all * (2.2 * steps - 22);
      p.better = 390 + want * (143 + 25 * odd) + shared * (48 - 4.4 * want) < margin * one;
    }
  };
  for (unsigned waves = 4; waves <= 8; waves += 4) choose(waves, 1, 3, 1.);
  if (p.splits == 1)
    for (unsigned waves = 4; waves <= 8; waves += 4) choose(waves, 4, 8, .75);
  return p;
}

}  // namespace qgemm_small_plan
}  // namespace tfcc_rocm
