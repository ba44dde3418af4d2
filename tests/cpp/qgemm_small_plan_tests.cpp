// The rule that deals small quantized products out over workgroups (wechat-tfcc_amd/csrc/qgemm_small_plan.hpp), on the host.
// Without arguments: its limits.  With some, groups of m n k batch: prints how many workgroups share a tile.  No GPU.
#include <cstdio>
#include <cstdlib>

#include "qgemm_small_plan.hpp"

using namespace tfcc_rocm::qgemm_small_plan;

static int failures = 0;
#define EXPECT(cond)                                         \
  do {                                                       \
    if (!(cond)) {                                           \
      ++failures;                                            \
      std::printf("FAIL line %d: %s\n", __LINE__, #cond);    \
    }                                                        \
  } while (0)

int main(int argc, char** argv) {
  if (argc > 1) {
    for (int i = 1; i + 3 < argc; i += 4) {
      const Plan p = plan_of(std::atoi(argv[i]), std::atoi(argv[i + 1]), std::atoi(argv[i + 2]), std::atoi(argv[i + 3]));
      std::printf("%u\n", p.better ? p.splits : 1u);
    }
    return 0;
  }
  EXPECT(plan_of(3, 910, 11304, 1).better && plan_of(32, 512, 8192, 1).better);
  // measured on both sides of the line: 1.2 to 1.35 times as long in several pieces; 0.86 and less
  EXPECT(!plan_of(526, 400, 1832, 1).better && !plan_of(1869, 32, 1824, 1).better && !plan_of(250, 200, 1624, 1).better);
  EXPECT(!plan_of(48, 4992, 1920, 1).better && !plan_of(194, 1152, 2048, 1).better);
  EXPECT(plan_of(105, 25, 2452, 1).better && plan_of(36, 467, 2486, 1).better && plan_of(133, 1144, 2187, 1).better);
  for (unsigned m = 1; m <= 3000; m = m * 5 / 4 + 1)
    for (unsigned n = 1; n <= 9000; n = n * 5 / 4 + 1)
      for (unsigned k = 1; k <= 20000; k = k * 4 / 3 + 1)
        for (unsigned batch = 1; batch <= 9; batch += 4) {
          const Plan p = plan_of(m, n, k, batch);
          const unsigned long long tiles = (unsigned long long)((m + 15) / 16) * ((n + 63) / 64) * batch;
          EXPECT(p.splits >= 1 && p.splits <= 32 && (p.splits == 1 || p.splitWaves == 4 || p.splitWaves == 8));
          EXPECT(p.splits > 1 || !p.better);
          // every word that workgroups meet in lies inside their piece of memory, and every workgroup has a step
          if (p.splits > 1) EXPECT(tiles * 16 * kCols <= kMaxResults && (p.splits - 1) * (p.splitWaves - 1) < (k + 63) / 64);
        }
  if (failures == 0) std::printf("qgemm small plan: all passed\n");
  return failures != 0;
}
