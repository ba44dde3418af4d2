// Which tiles the kernel of sgemm_deal.hip has for an fp32 product, over how many workgroups a tile's K is split, and about how long
// that takes.  Plain functions of integers, compiled for the dispatcher and for the tests.
#pragma once

namespace tfcc_rocm {
namespace sgemm_deal_plan {

constexpr unsigned kWaves = 8;              // of a workgroup, which deal the steps of K among themselves
constexpr unsigned kStep = 16;              // k of a step
constexpr unsigned kMaxParts = 1u << 20;    // results times splits of a product that is split, counted in whole tiles
constexpr unsigned kMaxSplits = 16;

struct Plan {
  unsigned splits, blocks;  // splits 0: not a product for this kernel; blocks of 32 columns in a tile of 32 rows
  double us;
};

inline unsigned long long tiles_of(unsigned m, unsigned n, unsigned blocks) {
  return (unsigned long long)((m + 31) / 32) * ((n + 32 * blocks - 1) / (32 * blocks));
}

// A constant, what the busiest CU does for its tiles (an XCD has a run of tiles with all their splits), and the meeting.  Fitted to
// 2600 launches of 220 products of 17 to 1024 rows, K from 768 to 8192, with weights and activations from the memory-side cache;
// met within 6 % on the average.
inline double microseconds(unsigned m, unsigned n, unsigned k, unsigned splits, unsigned blocks) {
  const unsigned long long tiles = tiles_of(m, n, blocks), busiest = ((tiles + 7) / 8 * splits + 31) / 32;
  const double thousands = k / (1000. * splits), filled = (tiles * splits < 256 ? tiles * splits : 256) / 256.;
  return 1.2 + busiest * (1.84 + .57 * blocks + thousands * (2.05 + 3.07 * blocks)) + .96 * filled * blocks * thousands +
         (splits > 1 ? 1.27 + .2 * splits * blocks : 0);
}

// The sizes that the fit covers; splits of 250 k and more, for shorter ones end before their loads have paid for the meeting.  In a
// stream that is being captured a tile of 32 x 32 has one workgroup, whatever the splits.  Fewer than 64 of them would gain as much launched,
// but the kernel of 16 x 16 tiles has four times as many there (286 x 8129 x 70 18 -> 15 us, captured 31 -> 60); more than 256 are a
// second round, and gain little launched: 24 products with 259 to 336 tiles took 0.92 of the tiled kernels' time launched and 1.42 captured (288 x
// 7296 x 920 52.8 -> 48.9, captured 54.3 -> 82.0).  160 products in between: launched 0.76 from cache and 0.62 with weights from memory, captured
// 1.04 and 0.92, 1.2 to 1.5 from cache those of up to some 2000 k (128 x 3072 x 768 15.1 -> 12.7, captured 15.7 -> 22.3; from memory 25.6 -> 13.1,
// captured 27.3 -> 27.8).
inline Plan plan_of(unsigned m, unsigned n, unsigned k) {
  Plan best{0, 1, 1e30};
  if (m < 17 || n < 32 || k < 768 || tiles_of(m, n, 1) < 64 || tiles_of(m, n, 1) > 256) return best;
  for (unsigned blocks = 1; blocks <= 2; ++blocks)
    for (unsigned s = 1; s <= kMaxSplits; ++s) {
      if (s > 1 && (k / s < 250 || tiles_of(m, n, blocks) * blocks * 1024 * s > kMaxParts)) break;
      const double us = microseconds(m, n, k, s, blocks);
      if (us < best.us) best = Plan{s, blocks, us};
    }
  return best;
}

}  // namespace sgemm_deal_plan
}  // namespace tfcc_rocm
