// Where the session cuts its uploads (wechat-tfcc_amd/host/upload_cut.h), on the host: every piece begins on a line, in the input as
// in the staging block, and all but an input's last are whole lines; nothing is lost; launches grow to their limit.  No GPU.
#include <cstdio>
#include <initializer_list>
#include <vector>

#include "upload_cut.h"

using tfcc::UploadCut;

static int failures = 0;
#define EXPECT(cond)                                         \
  do {                                                       \
    if (!(cond)) {                                           \
      ++failures;                                            \
      std::printf("FAIL line %d: %s\n", __LINE__, #cond);    \
    }                                                        \
  } while (0)

// as ROCMSession::upload goes through its inputs, with a staging block of `staging` bytes of which `used` are taken
static void upload(const std::vector<size_t>& inputs, size_t staging, size_t used) {
  UploadCut cut;
  size_t launch = 0, largest = 0;
  auto go = [&] {
    largest = launch > largest ? launch : largest;
    launch = 0;
    cut.launched();
  };
  for (size_t bytes : inputs) {
    size_t at = 0;
    while (at < bytes) {
      if (used >= staging) {
        if (launch > 0) go();
        used = 0;
      }
      const size_t n = cut.next(bytes - at, staging - used);
      EXPECT(n > 0 && at % UploadCut::kLine == 0 && used % UploadCut::kLine == 0 && (n % UploadCut::kLine == 0 || at + n == bytes));
      EXPECT(used + n <= staging);
      if (n == 0) return;
      used += UploadCut::padded(n);
      at += n;
      launch += UploadCut::padded(n);
      if (cut.put(n)) go();
    }
    EXPECT(at == bytes);
  }
  EXPECT(largest <= size_t(768) << 10);
}

int main() {
  const size_t mb = size_t(1) << 20;
  upload({301 * 4, 301 * 768 * 4}, 4 * mb, 0);  // a mask in front of the hidden states
  upload({77 * 4, 3 * mb}, 4 * mb, 0);
  upload({77 * 4, 384 * 1024, 768 * 1024 + 12, 20}, 2 * mb, 0);
  for (size_t first : {size_t(1), size_t(4), size_t(63), size_t(64), size_t(65), size_t(116), size_t(1204), size_t(384) * 1024 - 1, size_t(384) * 1024 + 1})
    for (size_t second : {size_t(1), size_t(383) * 1024, size_t(384) * 1024, mb, 5 * mb + 3})
      for (size_t staging : {size_t(256) << 10, mb, 8 * mb})
        for (size_t used : {size_t(0), size_t(64), staging - 64, staging}) {
          upload({first, second}, staging, used);
          upload({second, first, second, first, first}, staging, used);
        }
  upload(std::vector<size_t>(1000, 777), mb, 0);
  if (failures == 0) std::printf("upload cut: all passed\n");
  return failures != 0;
}
