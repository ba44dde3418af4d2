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

// Whether there is enough work for the form of any alignment, in wavefronts of 64 x 256.  Against the kernel for small products of any
// alignment, us: 7900 x 5814 20.8 -> 12.6, 5799 x 9800 20.1 -> 13.4, with exact sums 2448 x 4782 8.6 -> 7.3, 2052 x 3704 7.8 -> 6.4, 10124 x
// 1235 9.4 -> 7.8.  Below the line 6 x 2432 x 7191 8.8 -> 9.3, 2 x 924 x 11952 6.5 -> 6.7, 8 x 4040 x 6689 10.9 -> 11.5, with exact sums 6 x
// 1766 x 5686 6.5 -> 7.1, 4 x 883 x 10148 5.4 -> 6.4 (a K that short is read at once there too), 5 x 4516 x 2543 6.2 -> 7.5.  With sixteen
// wavefronts to a workgroup, from 1400 on, so few of them leave CUs without work, and rows at odd addresses take a CU's load path twice as
// long: 32 products of 1400 to 2100 took 0.86 to 1.26 of the time there, none gained on the average (5 x 2299 x 10293 8.4 -> 10.0, 6 x 11815 x 1839
// 9.1 -> 10.6), 17 without exact sums of 1400 to 1700 0.97 (8 x 2024 x 11368 7.4 -> 8.8); from 2100 on 0.8 (4 x 4002 x 8635 0.74).
inline bool ragged_pays(unsigned n, unsigned k, bool exact) {
  const unsigned long long work = (unsigned long long)((n + kCols - 1) / kCols) * ((k + 63) / 64);
  if (!exact) return work >= (n % 4 == 0 ? 1700u : 2100u);
  return n % 4 == 0 ? work >= 420 : work >= 2100 || (work >= 720 && work < 1400);
}

}  // namespace gemv_wide_plan
}  // namespace tfcc_rocm
