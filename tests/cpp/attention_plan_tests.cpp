// Which attention kernel takes a call (wechat-tfcc_amd/csrc/attention_plan.hpp), on the host: the rule's lines, and that no call has more
// threads than a launch may have where blocks of 64 rows, which take any, would not.  No GPU.
#include <cstdio>
#include <initializer_list>

#include "attention_plan.hpp"

using namespace tfcc_rocm::attention_plan;

static int failures = 0;
#define EXPECT(cond)                                         \
  do {                                                       \
    if (!(cond)) {                                           \
      ++failures;                                            \
      std::printf("FAIL line %d: %s\n", __LINE__, #cond);    \
    }                                                        \
  } while (0)

int main() {
  EXPECT(kernel_of(29, 29, 12, 256) == kRows16 && kernel_of(64, 64, 1536, 256) == kRows16 && kernel_of(128, 128, 24, 256) == kRows16);
  EXPECT(kernel_of(16, 100, 480, 256) == kRows16 && kernel_of(128, 128, 96, 256) == kRows64 && kernel_of(128, 128, 192, 256) == kRows32);
  EXPECT(kernel_of(512, 512, 96, 256) == kRuns32 && kernel_of(384, 384, 12, 256) == kRuns16);
  for (unsigned s : {1u, 9u, 16u, 17u, 32u, 33u, 48u, 64u, 65u, 97u, 128u, 1000u, 4096u})
    for (unsigned t : {1u, 29u, 64u, 65u, 128u, 129u, 512u})
      for (unsigned long long heads = 2; heads < 1ull << 24; heads = heads * 3 / 2 + (heads & 1)) {
        if (launchable(s, heads, kRows64) && launchable(s, heads, kRows32)) EXPECT(launchable(s, heads, kernel_of(s, t, heads, 256)));
      }
  // 2^28 rows: the first that are too many for blocks of 16
  EXPECT(kernel_of(64, 64, 1u << 22, 256) != kRows16 && kernel_of(64, 64, (1u << 22) - 2, 256) == kRows16);
  EXPECT(launchable(64, 1u << 22, kernel_of(64, 64, 1u << 22, 256)));
  if (failures == 0) std::printf("attention plan: all passed\n");
  return failures != 0;
}
