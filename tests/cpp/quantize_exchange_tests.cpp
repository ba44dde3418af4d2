// The words of the one-launch quantize (wechat-tfcc_amd/csrc/quantize_exchange.hpp), on the host: no word of another call, however
// many calls ago, and none that nobody has written is taken for this call's.  No GPU.
#include <cstdio>
#include <initializer_list>

#include "quantize_exchange.hpp"

using namespace tfcc_rocm::quantize_exchange;

static int failures = 0;
#define EXPECT(cond)                                         \
  do {                                                       \
    if (!(cond)) {                                           \
      ++failures;                                            \
      std::printf("FAIL line %d: %s\n", __LINE__, #cond);    \
    }                                                        \
  } while (0)

int main() {
  for (unsigned long long call : {0ull, 1ull, 255ull, 65535ull, (1ull << 32) - 2, (1ull << 32) - 1, 1ull << 32, (1ull << 47) + 5, kNumbers - 2}) {
    const unsigned long long number = number_of(call);
    EXPECT(number != 0 && number < kNumbers);
    EXPECT(!belongs_to(0, number));
    for (unsigned long long apart : {1ull, 256ull, 1ull << 16, 1ull << 32, 1ull << 33, 256ull << 32, 1ull << 47})  // 256: the sets of words
      EXPECT(number_of(call + apart) != number && !belongs_to(word_of(number, 0x3f800000u, true), number_of(call + apart)));
    for (unsigned value : {0u, 0x80000000u, 0x0000ffffu, 0xffff0000u, 0x7f7fffffu, 0xff800000u, 0xffffffffu}) {
      const unsigned long long low = word_of(number, value, false), high = word_of(number, value, true);
      EXPECT(belongs_to(low, number) && belongs_to(high, number) && value_of(low, high) == value);
    }
  }
  if (failures == 0) std::printf("quantize exchange: all passed\n");
  return failures != 0;
}
