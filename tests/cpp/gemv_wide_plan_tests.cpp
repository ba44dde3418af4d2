// How the K of an int8 product of up to eight rows is dealt out (wechat-tfcc_amd/csrc/gemv_wide_plan.hpp), on the host: no GPU.
#include <cstdio>
#include <initializer_list>

#include "gemv_wide_plan.hpp"

using namespace tfcc_rocm::gemv_wide_plan;

static int failures = 0;
#define EXPECT(cond)                                         \
  do {                                                       \
    if (!(cond)) {                                           \
      ++failures;                                            \
      std::printf("FAIL line %d: %s\n", __LINE__, #cond);    \
    }                                                        \
  } while (0)

int main() {
  // few wavefronts: eight to a workgroup where their parts may meet
  EXPECT(plan_of(8192, 1024, false, true).waves == 8 && plan_of(8192, 1024, false, true).parts == 2);
  // where they may not, sixteen have a short K alone
  EXPECT(plan_of(8192, 1024, false, false).waves == 16 && plan_of(8192, 1024, false, false).parts == 1);
  for (unsigned n = 256; n <= 70000; n += 4080)
    for (unsigned k = 16; k <= 40000; k = k * 5 / 4 + 16)
      for (int ragged = 0; ragged < 2; ++ragged) {
        const Plan with = plan_of(n, k, ragged, true), without = plan_of(n, k, ragged, false);
        const unsigned steps = (k + 63) / 64;
        const unsigned long long blocks = (n + kCols - 1) / kCols;
        for (const Plan& p : {with, without}) {
          EXPECT((unsigned long long)p.waves * p.stepsPerWave * p.parts >= steps);
          EXPECT((unsigned long long)p.waves * p.stepsPerWave * (p.parts - 1) < steps);
          EXPECT(p.waves == 4 || p.stepsPerWave == 1);
        }
        // what sixteen wavefronts cover needs no workspace, and what they do not cover is the same with and without
        if (steps <= 16 && blocks <= 1024) EXPECT(without.parts == 1);
        else EXPECT(with.waves == without.waves && with.stepsPerWave == without.stepsPerWave && with.parts == without.parts);
      }
  // any alignment: rows at odd addresses not while sixteen wavefronts to a workgroup leave CUs without work, nor just above the least work
  EXPECT(!ragged_pays(10293, 2299, true) && !ragged_pays(1839, 11815, true) && !ragged_pays(2543, 4516, true) && !ragged_pays(11368, 2024, false));
  EXPECT(ragged_pays(4782, 2448, true) && ragged_pays(9271, 2352, true) && ragged_pays(8635, 4002, true) && ragged_pays(5814, 7900, false) &&
         ragged_pays(3704, 2052, true) && ragged_pays(11368, 2024, true));
  std::printf(failures ? "%d failures\n" : "all passed\n", failures);
  return failures != 0;
}
