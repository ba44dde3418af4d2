// Host-side test of the rule that picks LSTM sequences for one launch (wechat-tfcc_amd/csrc/lstm_sequence_plan.hpp): a GPU with
// fewer CUs than the launch has workgroups gets no workspace, which sends the caller to the step-by-step form.  No GPU.
#include <cstdio>
#include <initializer_list>

#include "lstm_sequence_plan.hpp"

using namespace tfcc_rocm::lstm_plan;

static int failures = 0;
#define EXPECT(cond)                                         \
  do {                                                       \
    if (!(cond)) {                                           \
      ++failures;                                            \
      std::printf("FAIL line %d: %s\n", __LINE__, #cond);    \
    }                                                        \
  } while (0)

int main() {
  EXPECT(workspace_bytes(16, 1024, 2, 256) == 2u * 2 * 16 * 1024 * 8 + 64);
  EXPECT(workspace_bytes(1, 1, 1, 1) == 2u * 256 * 8 + 64);
  EXPECT(workspace_bytes(0, 64, 2, 256) == 0 && workspace_bytes(17, 64, 2, 256) == 0);
  EXPECT(workspace_bytes(1, 0, 2, 256) == 0 && workspace_bytes(1, 1025, 2, 256) == 0);
  EXPECT(workspace_bytes(1, 64, 0, 256) == 0 && workspace_bytes(1, 64, 3, 256) == 0);
  for (int cus : {-1, 0, 1, 32, 64, 128, 255, 256})
    for (unsigned directions = 1; directions <= 2; ++directions)
      for (unsigned units = 1; units <= 1024; ++units) {
        unsigned needed = 0;
        for (unsigned d = 0; d < directions; ++d)
          for (unsigned u = 0; u < units; u += 8) ++needed;
        EXPECT((workspace_bytes(4, units, directions, cus) != 0) == (cus > 0 && needed <= (unsigned)cus));
      }
  for (unsigned directions = 1; directions <= 2; ++directions)
    for (unsigned batch = 1; batch <= 16; ++batch)
      for (unsigned units = 1; units <= 1024; ++units) {
        const unsigned rows = rows_of_xcd(batch, units, directions, 256);
        EXPECT((rows != 0) == (units <= 768));
        EXPECT(rows_of_xcd(batch, units, directions, 128) == 0);
        if (rows == 0) continue;
        const unsigned groups = (batch + rows - 1) / rows, each = 8 * ((units + 255) / 256);
        EXPECT(rows <= 4 && groups * directions <= kXcds && (units + each - 1) / each <= kCusOfXcd);
        // two sets of 64-bit words with this form's pitch fit in front of the flag
        const size_t pitch = (units + 255) / 256 * 256;
        EXPECT(2 * directions * batch * pitch * 8 + 64 <= workspace_bytes(batch, units, directions, 256));
      }
  if (failures == 0) std::printf("lstm plan: all passed\n");
  return failures != 0;
}
