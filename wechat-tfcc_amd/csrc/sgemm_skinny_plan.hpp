// Which fp32 products take the kernel for few rows (sgemm_skinny.hip), in which tiles and over how many workgroups, and which the one
// whose tiles have a dealt K (sgemm_deal.hip).  Plain functions of integers, compiled for the dispatcher and for the tests.
#pragma once

#include "sgemm_deal_plan.hpp"
#include "sgemm_tiles.hpp"

namespace tfcc_rocm {
namespace sgemm_skinny_plan {

constexpr unsigned kMaxParts = 1024;  // blocks of 16 x 16 x splits of a product that is split

struct Plan {
  unsigned splits, rows;  // workgroups that share a tile's K; blocks of sixteen rows in a tile
  bool better;            // than the other kernels
  double us;
  bool unsplit;           // tiles of sixteen rows fill the chip without splits
};

// Whether a product takes this kernel, and over how many workgroups a tile's K is split: from the sizes of one product
// alone, so that it is summed the same way alone, in a group and with B transposed.  Nanoseconds as measured, launch aside:
// a CU takes 2.8 per k of every tile it has; arriving and adding up costs 1300 and 200 more per split; the 32-row tiles with
// four K groups take 5.1 per k while there is one for each CU.  (The line stands at 4.6, so that what is in doubt stays
// where it was.)  Splits of less than 512 k end before their loads have paid for the arrival: 2048 -> 512 with 9 rows, 7.4 us in
// splits of 256 against 6.2.  Below 256 k nothing is split in the tiled kernels either, and a product of more than eight rows keeps
// their bits, which are those it has in a batch.
//
// Up to eight rows the other kernel is the streaming one (sgemv.hip), which has a CU for 32 columns and walks what K has
// beyond a multiple of 64 eight rows at a time.  See takes_few_rows.
//
// More than sixteen rows have tiles of 32 as well, which read B once for two blocks of rows, one workgroup to a CU: they are taken
// where the times below, fitted to 900 launches of 170 products of 17 to 100 rows and met within 5 %, say so.  Against the tiled kernels,
// whose estimate is met without a remainder and from cache (1.19 of it with weights from memory, 1.27 with a K or an N that is no
// multiple of their pieces), and against tiles of 16: 26 x 1328 x 3072 10.7 -> 8.4 us, 18 x 1006 x 3222 8.6 -> 6.7, 29 x 768 x 3072
// 7.1 -> 6.1, 41 x 968 x 1952 8.3 -> 7.1, 94 x 3048 x 400 10.2 -> 9.0.  A CU takes one such workgroup, and an XCD has a run of tiles with
// all their splits: 84 tiles in three splits are 33 workgroups on 32 CUs (17 x 3163 x 1336 12.3 us, 8.7 in tiles of 16; 211 x 1903 x 192 9.5
// and 6.3).
//
// The tiled kernels' estimate lies between weights from cache and from memory, and tiles without a remainder take 0.78 of it from cache.  Two
// blocks gain from memory, where there are many weights; with few columns there are not, and past 1024 k the rows no longer stay in the L2 of
// every XCD either: 960 x 1120 x 128 6.5 -> 8.7 us (with weights from memory 7.6 -> 8.6), 674 x 1344 x 144 7.5 -> 8.9 (9.9 -> 9.0), 754 x 1216 x 136 7.1
// -> 8.6 from cache.  Those stay with the tiled kernels.  More columns: 51 x 1152 x 1408 6.8 -> 7.3 (12.0 -> 8.7), 17 x 1216 x 2944 7.4 ->
// 6.3 (12.3 -> 8.7).

// Up to eight rows: here or in the streaming kernel.  300 products, replayed with weights from memory / from cache, streaming -> here: 8 x
// 64 x 2048 3.8/3.6 -> 2.2/2.1 us, 4 x 496 x 302 11.4/6.1 -> 3.1/2.7, 8 x 832 x 960 5.3/4.8 -> 3.8/3.4, 1 x 424 x 1588 4.3/3.0 ->
// 3.1/2.7; launched, 4 x 3072 x 768 12.0/8.0 -> 6.6/6.4, 1 x 8192 x 2048 20.5 -> 14.6, 8 x 2304 x 4000 14.0/11.0 -> 9.9/8.0.
// The streaming kernel keeps one row of up to 1024 k, a multiple of its chunks of 64 (1 x 960 x 128 3.5/2.9, here 3.5/3.3; 1 x 192 x 966
// 2.7/2.35, here 2.4/2.2, but its launch, which is the longer part, costs the host 0.15 less), and what reads
// whole lines of B on most of the CUs, but for a short K: 1 x 5120 x 5120 27, here 34, 4 x 1024 x 5376 6.5/6.0, here 8.6/7.8, 4 x 4096
// x 11008 36, here 47; 6 x 192 x 9216 6.4/5.7 -> 4.0/3.6, 2 x 16 x 5984 2.9/2.5 -> 2.4/2.3.  Other widths come here (4 x 1024 x 7100 10.6 -> 8.3,
// 1 x 3000 x 7100 24 -> 16), and so do more than two rows of a K with a rest (4 x 700 x 6144 13.8 -> 7.0), except of wide and deep ones, which
// the memory decides and 64-byte pieces do not suit (2 x 2000 x 15000 25, here 28, 4 x 4096 x 11000 39, here 45; 4 x 1000 x 16001 15.9 -> 13.2).
// One and two rows of whole chunks stay there too where splitting K does not pay.  Few columns: two or three splits of up to 1600 k meet for
// longer than they save (1 x 1472 x 64 launched 4.1 -> 4.8 us and replayed 3.9 -> 5.2, with weights from memory 4.4 -> 4.7 and 4.4 -> 5.2; from
// 768 columns on memory decides, 1 x 1472 x 768 4.5 -> 4.7 and 6.9 -> 5.3).  And a B of 20 to 32 MB in whole lines, which the L2s of the eight
// XCDs hold together and the streaming kernel reads in turn (1 x 2048 x 3840 launched 5.1 -> 7.0, from memory 11.5 -> 11.0; with fewer
// columns there is more to gain from memory, 1 x 2304 x 2304 5.5 -> 5.9 and 11.2 -> 8.3).
inline bool takes_few_rows(unsigned m, unsigned n, unsigned k) {
  if (n <= 4096) {
    if (m > 2 || k % 64 != 0) return true;
    if (k > 1152 && k <= 1600 && n <= 640) return false;
    const unsigned long long words = (unsigned long long)k * n;
    if (n % 128 == 0 && n >= 2688 && words > 5400000 && words < 8000000) return false;
    return m > 1 || k > 1024;
  }
  if (n % 32 != 0 || (k % 64 != 0 && m > 2)) return n < 10240 || k <= 1600;
  return n < 10240 && k <= (m > 4 ? 512u : m > 2 ? 256u : 128u);
}

// What the dealt kernel has to be thought to take less than, to be taken instead of the tiled ones.  Their estimate lies between weights
// from cache and from memory.  Tiles without a remainder and with a short K are nearer to the former, 0.78 of it, while weights from memory are
// what the dealt kernel gains most from; with few columns there are not many weights, and what would be lost counts: with a line
// at 0.97 as for wider ones, launched from cache / memory and replayed from cache / memory, 398 x 1344 x 208 took 1.11/0.85 and 1.40/1.10 of
// the tiled kernels' time, 332 x 1664 x 344 1.07/0.80 and 1.41/1.07, 896 x 2048 x 124 1.09/0.78 and 1.42/1.07; 128 x 1344 x 768, where both are
// thought to be equal, 1.10/0.83 and 1.42/1.02.
inline double dealt_below(unsigned m, unsigned n, unsigned k) {
  const double tiled = sgemm_tiles::microseconds(m, n, k, 1);
  if (tiled >= 15 || k % 32 != 0 || n % 4 != 0) return tiled;
  return 2 * m > n ? .84 * tiled : .97 * tiled;
}

// deal: what sgemm_deal_plan.hpp has for the same product.
inline Plan plan_of(unsigned m, unsigned n, unsigned k, const sgemm_deal_plan::Plan& deal) {
  const unsigned long long tiles = (unsigned long long)((m + 15) / 16) * ((n + 15) / 16);
  if (k < (m > 8 ? 256u : 16u) || tiles > kMaxParts) return Plan{1, 1, false, 0, false};
  Plan best{1, 1, false, 0, false};
  unsigned long long bestCost = ~0ull;
  for (unsigned s = 1; s == 1 || (s <= k / 512 && tiles * s <= kMaxParts); ++s) {
    const unsigned long long perCu = (tiles * s + 255) / 256;
    const unsigned long long cost = perCu * k * 28 / s + (s > 1 ? 13000 + 2000 * s : 0);
    if (cost < bestCost) {
      best.splits = s;
      bestCost = cost;
    }
  }
  best.us = 2.5 + bestCost * 1e-4;
  best.better = m > 8 ? bestCost < (unsigned long long)k * 46 : takes_few_rows(m, n, k);
  if (m <= 16) return best;
  best.unsplit = best.better && best.splits == 1;
  double line = .92 * best.us;
  if (!best.better) {
    const double tiled = sgemm_tiles::microseconds(m, n, k, 1);
    line = (k % 32 != 0 || n % 4 != 0 ? 1.15 : 2 * m > n && k > 1024 ? .78 : 1.05) * tiled;
    if (deal.splits > 0 && deal.us < dealt_below(m, n, k) && .9 * deal.us < line) line = .9 * deal.us;  // the one that takes it otherwise
  }
  for (unsigned rows = best.better ? 2 : 1; rows <= 2; ++rows) {
    const unsigned long long count = (unsigned long long)((m + 16 * rows - 1) / (16 * rows)) * ((n + 15) / 16);
    for (unsigned s = 1; s == 1 || s <= k / 512; ++s) {
      if (count * rows * s > kMaxParts) break;
      const double perCu = (double)(rows == 1 ? (count * s + 255) / 256 : ((count + 7) / 8 * s + 31) / 32);
      const double filled = count * s / 256., thousands = k / (1000. * s);
      const double us = rows == 1 ? 2.94 + perCu * (2.04 * thousands + .2) + .39 * filled * thousands + (s > 1 ? .07 + .38 * s : 0)
                                  : 1.66 + perCu * (3.52 * thousands + 1.19) + .97 * filled * thousands + (s > 1 ? .66 + .28 * s : 0);
      if (us < line) {
        line = us;
        best = Plan{s, rows, true, us, best.unsplit};
      }
    }
  }
  return best;
}

enum Kernel { kOther, kSkinny, kDeal };
struct Choice {
  Kernel kernel;
  Plan skinny;
  sgemm_deal_plan::Plan deal;
};

// Which of the two kernels whose workgroups share a K: the one for tiles of 32 rows where it is thought to be faster than the
// other by a tenth, or than the tiled kernels at all.  Of 220 products of 17 to 1024 rows and 768 k and more it takes 47,
// at 0.79 of the time (up to 1.0), another 13 lose a tenth without it.  What the bf16 matrix ops take stays there (bf16, asked for
// where it matters), and so does what fills the chip in tiles of 16 without splits: launched it would gain a quarter, but replayed, when
// the dealt kernel has a CU for a tile, take 1.8 of the time (485 x 4448 x 104 16.5 us, dealt 12.5 launched and 29.9 replayed).
template <class Asked>
inline Choice choose(unsigned m, unsigned n, unsigned k, const Asked& bf16) {
  Choice c{kOther, {1, 1, false, 0, false}, sgemm_deal_plan::plan_of(m, n, k)};
  c.skinny = plan_of(m, n, k, c.deal);
  if (c.skinny.better) c.kernel = kSkinny;
  if (c.deal.splits > 0 && !c.skinny.unsplit &&
      c.deal.us < (c.skinny.better ? .9 * c.skinny.us : bf16() ? 0 : dealt_below(m, n, k)))
    c.kernel = kDeal;
  return c;
}

}  // namespace sgemm_skinny_plan
}  // namespace tfcc_rocm
