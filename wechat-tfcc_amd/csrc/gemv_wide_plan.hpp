// How the K of an int8 product of up to eight rows is dealt out (gemv_u8s8_wide.hip).  A plain function of integers, compiled for the
// launcher and for the tests.
#pragma once

namespace tfcc_rocm {
namespace gemv_wide_plan {

constexpr int kCols = 256;  // columns of a workgroup

struct Plan {
  unsigned waves;         // of a workgroup
  unsigned stepsPerWave;  // of 64 rows of B
  unsigned parts;         // workgroups that share a column block's K: more than one meet in a workspace
};

// Sixteen wavefronts make one step each; a product that would need more than about four such workgroups for each CU goes to four
// wavefronts of several steps.
//
// Sixteen wavefronts of one step leave most CUs without work while there are few, and a workgroup's bytes go through one CU: eight
// of them, us: 1984 x 5056 7.6 -> 6.3, 3200 x 2688 7.6 -> 6.5, 1344 x 9792 7.8 -> 6.7; past 900 wavefronts 6336 x 2560 7.2 -> 7.6, 5760 x
// 9792 12.8 -> 13.8.  Ragged loads take a CU longer: 2104 x 9276 8.3 -> 7.9, 5789 x 3292 8.9 -> 8.5, 3024 x 8698 9.5 -> 9.9.  (Four:
// more parts to add up, 1984 x 5056 7.6, 1344 x 9792 7.8.)
//
// meets: whether the launch has a workspace to itself.  Without one a K of up to sixteen steps stays in one part.
inline Plan plan_of(unsigned n, unsigned k, bool ragged, bool meets) {
  const unsigned long long blocks = (n + kCols - 1) / kCols;
  const unsigned steps = (k + 63) / 64;
  Plan p{16, 1, 0};
  if (blocks * ((steps + 15) / 16) > 1024) p.waves = 4, p.stepsPerWave = 4;
  while (blocks * ((steps + p.waves * p.stepsPerWave - 1) / (p.waves * p.stepsPerWave)) > 1024 && p.stepsPerWave < 64) p.stepsPerWave *= 2;
  if (p.stepsPerWave == 1 && blocks * steps < (ragged ? 1400u : 900u) && (meets || steps > 16)) p.waves = 8;
  p.parts = (steps + p.waves * p.stepsPerWave - 1) / (p.waves * p.stepsPerWave);
  return p;
}

}  // namespace gemv_wide_plan
}  // namespace tfcc_rocm
