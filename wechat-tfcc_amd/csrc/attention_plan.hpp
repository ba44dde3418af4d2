// Which kernel of attention.hip takes a call.  A plain function of integers, compiled for the dispatcher and for the tests.
#pragma once

namespace tfcc_rocm {
namespace attention_plan {

constexpr unsigned kWholeKeys = 128;  // keys up to which the scores of a row block are in one piece

// kRows64, kRows32, kRows16: query rows per workgroup, scores in one piece; kRuns16, kRuns32: keys in runs of 32
enum Kernel { kRows64, kRows32, kRows16, kRuns16, kRuns32 };
constexpr unsigned rows_of(Kernel kernel) { return kernel == kRows64 ? 64 : kernel == kRows32 || kernel == kRuns32 ? 32 : 16; }
constexpr unsigned threads_of(Kernel kernel) { return kernel == kRows64 ? 512 : 256; }
constexpr unsigned long long blocks_of(unsigned s, unsigned long long heads, unsigned rows) { return (s + rows - 1) / rows * heads; }
// A launch has fewer than 2^32 threads (the workgroups are rounded up to a multiple of eight).
constexpr bool launchable(unsigned s, unsigned long long heads, Kernel kernel) {
  return (blocks_of(s, heads, rows_of(kernel)) + 7) / 8 * 8 * threads_of(kernel) < 1ull << 32;
}

inline Kernel kernel_of(unsigned s, unsigned t, unsigned long long heads, int cus) {
  const unsigned long long blocks64 = blocks_of(s, heads, 64), blocks32 = blocks_of(s, heads, 32), blocks16 = blocks_of(s, heads, 16);
  // More than 128 keys: two blocks of 16 rows share the loads of K and V where there are six or more for each CU (8 x 12 heads of 512
  // rows 72.8 -> 68.4 us, 16 x 12 of 384 86.0 -> 79.5, 8 x 12 of 384 45.7 -> 46.1); with fewer they fill the GPU less evenly (4 x 12
  // of 384 27.2 -> 29.3, 12 of 1024 35.9 -> 43.8, 12 of 256 6.7 -> 9.6).
  if (t > kWholeKeys) return blocks16 < 6ull * cus ? kRuns16 : kRuns32;
  // Blocks of 16 rows: up to 64 keys always (128 x 12 heads of 64 rows 37.1 -> 33.7 us, 32 x 12 12.3 -> 12.4, 64 x 12 of 32 11.2 -> 10.6).  Beyond, every
  // block walks twice the keys, which is faster where there are no more blocks than CUs or no more than with 32 rows
  // (2 x 12 heads of 128 rows 7.9 -> 6.2 us, 40 x 12 of 16 rows and 100 keys 10.4 -> 8.7), and not otherwise (4 x 12 of 100
  // rows 7.7 -> 8.4, 8 x 12 of 128 10.4 -> 11.6).  They have twice the threads of blocks of 64 rows, which from 2^28 rows on are
  // more than a launch may have.
  if ((t <= 64 || s <= 16 || blocks16 <= (unsigned long long)cus) && launchable(s, heads, kRows16)) return kRows16;
  // A CU works through its blocks roughly one after the other (two resident workgroups overlap little: 19.1 us for
  // 384 blocks of 64 rows against 12.7 for 192), so what counts is the largest number of rows any CU gets; a block of
  // 32 rows costs about 0.55 of a block of 64 (K and V are loaded per block).  16 x 12 heads of 128 rows: 17.8 against
  // 19.1 us with 32 rows; 32 x 12 heads: 30.5 against 27.7, so those keep 64.
  const unsigned long long perCu64 = (blocks64 + cus - 1) / cus, perCu32 = (blocks32 + cus - 1) / cus;
  return perCu32 * 55 < perCu64 * 100 ? kRows32 : kRows64;
}

}  // namespace attention_plan
}  // namespace tfcc_rocm
