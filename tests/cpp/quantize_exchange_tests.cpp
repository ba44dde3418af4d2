// The words of the one-launch quantize (wechat-tfcc_amd/csrc/quantize_exchange.hpp), on the host: no word of another call, however
// many calls ago, and none that nobody has written is taken for this call's; and that every workgroup has a CU,
// beside those of other streams too.  No GPU.
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
  for (int cus : {-1, 0, 1, 32, 64, 128, 255, 256, 304})
    for (unsigned long long total : {1ull, 4096ull, 4097ull, 40961ull, 32ull * 4096, 128ull * 4096, 128ull * 4096 + 1, 1ull << 20, (1ull << 20) + 1,
                                     4ull << 20, (4ull << 20) + 1, 8ull << 20, (8ull << 20) + 1, 1ull << 40}) {
      const unsigned quads = quads_of(total, cus), room = cus <= 0 ? 0 : cus < 256 ? cus : 256;
      if (quads == 0) EXPECT(total > 8ull * kPiece * room);
      else EXPECT(workgroups(total, quads) <= room && workgroups(total, quads) * quads * kPiece >= total && (quads == 1 || workgroups(total, quads / 2) > room));
    }
  int streams[9];
  for (unsigned count : {1u, 2u, 3u, 4u, 8u, 9u}) {  // in turn
    LastStreams last;
    for (unsigned call = 0; call < 100; ++call) {
      const unsigned seen = last.with(streams + call % count), most = call + 1 < 8 ? call + 1 : 8;
      EXPECT(seen == (count < most ? count : most));
      if (call >= 7 && count > 2) EXPECT(seen > streams_of(4) && seen > streams_of(8) && seen <= streams_of(1));
      if (call >= 7 && count <= 2) EXPECT(seen <= streams_of(8));
    }
    for (unsigned call = 0; call < 20; ++call) {  // the others have ended
      const unsigned seen = last.with(streams);
      EXPECT(call < 7 || seen == 1);
    }
  }
  if (failures == 0) std::printf("quantize exchange: all passed\n");
  return failures != 0;
}
