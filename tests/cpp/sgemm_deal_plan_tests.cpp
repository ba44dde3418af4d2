// The plan of fp32 products whose K is dealt out over wavefronts and workgroups (wechat-tfcc_amd/csrc/sgemm_deal_plan.hpp), on the
// host.  Without arguments: its limits.  With some, groups of m n k: prints the splits and blocks of each product.  No GPU.
#include <cstdio>
#include <cstdlib>

#include "sgemm_deal_plan.hpp"

using namespace tfcc_rocm::sgemm_deal_plan;

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
    for (int i = 1; i + 2 < argc; i += 3) {
      const Plan p = plan_of(std::atoi(argv[i]), std::atoi(argv[i + 1]), std::atoi(argv[i + 2]));
      std::printf("%u %u\n", p.splits, p.blocks);
    }
    return 0;
  }
  for (unsigned m = 1; m <= 5000; m = m * 5 / 4 + 1)
    for (unsigned n = 1; n <= 9000; n = n * 5 / 4 + 1)
      for (unsigned k = 1; k <= 70000; k = k * 5 / 4 + 1) {
        const Plan p = plan_of(m, n, k);
        if (p.splits == 0) continue;
        // K of at least a step, splits of at least a few, and the partial tiles within the memory in which they meet
        EXPECT(m > 16 && n >= 32 && k >= 768 && p.splits <= kMaxSplits && (p.blocks == 1 || p.blocks == 2));
        EXPECT(p.splits == 1 || (k / p.splits >= 250 && tiles_of(m, n, p.blocks) * p.blocks * 1024 * p.splits <= kMaxParts));
        EXPECT(p.us == microseconds(m, n, k, p.splits, p.blocks));
      }
  EXPECT(plan_of(75, 832, 3072).splits == 3 && plan_of(96, 824, 7608).blocks == 2);
  EXPECT(plan_of(16, 832, 3072).splits == 0 && plan_of(75, 832, 767).splits == 0 && plan_of(2048, 2048, 2048).splits == 0);
  if (failures == 0) std::printf("sgemm deal plan: all passed\n");
  return failures != 0;
}
