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

// The sizes that the fit covers; splits of 250 k and more, for shorter ones end before their loads have paid for the meeting.  Fewer
// than 64 tiles of 32 x 32 would gain as much, but not in a stream that is being captured, where a tile has one workgroup and the
// kernel of 16 x 16 tiles four times as many (286 x 8129 x 70 18 -> 15 us, captured 31 -> 60).
inline Plan plan_of(unsigned m, unsigned n, unsigned k) {
  Plan best{0, 1, 1e30};
  if (m < 17 || n < 32 || k < 768 || tiles_of(m, n, 1) < 64 || tiles_of(m, n, 1) > 700) return best;
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
