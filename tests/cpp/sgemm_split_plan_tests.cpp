// The rule that sends fp32 products to the kernels on the bf16 matrix cores (wechat-tfcc_amd/csrc/sgemm_split_plan.hpp), on the
// host.  Without arguments: its limits.  With some, groups of m n k batch: prints the kernel that takes each product.  No GPU.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "sgemm_split_plan.hpp"

using namespace tfcc_rocm::sgemm_split_plan;

static int failures = 0;
#define EXPECT(cond)                                         \
  do {                                                       \
    if (!(cond)) {                                           \
      ++failures;                                            \
      std::printf("FAIL line %d: %s\n", __LINE__, #cond);    \
    }                                                        \
  } while (0)

static int plain(unsigned m, unsigned n, unsigned k, unsigned batch = 1, bool transB = false) {
  return kernel_of(m, n, k, k, transB ? k : n, n, transB, batch);
}

int main(int argc, char** argv) {
  if (argc > 1) {
    for (int i = 1; i + 3 < argc; i += 4)
      std::printf("%d\n", plain(std::atoi(argv[i]), std::atoi(argv[i + 1]), std::atoi(argv[i + 2]), std::atoi(argv[i + 3])));
    return 0;
  }
  EXPECT(plain(4096, 4096, 4096) == kWide && plain(2048, 2048, 2048) == k128 && plain(1024, 1024, 2048) == k64);
  for (unsigned m : {1u, 8u, 47u, 4096u})  // few rows, few columns, short K, few tiles: the fp32 matrix ops
    EXPECT(plain(m, 47, 4096) == kNone && plain(47, m, 4096) == kNone && plain(m, 4096, 127) == kNone && plain(m, 64, 4096) == kNone);
  EXPECT(plain(64, 127 * 64, 8192) == kNone && plain(512, 512, 191, 64) == kNone);
  // the reach of the kernels' 32-bit byte offsets
  EXPECT(kernel_of(4096, 4096, 4096, (1u << 29) / (4096 + 256) + 1, 4096, 4096, false, 1) == kNone);
  EXPECT(kernel_of(4096, 4096, 4096, 4096, (1u << 29) / (4096 + 256) + 1, 4096, false, 1) == kNone);
  EXPECT(kernel_of(4096, 4096, 4096, 4096, (1u << 29) / (4096 + 256) + 1, 4096, true, 1) == kNone);
  EXPECT(kernel_of(4096, 4096, 4096, 4096, 4096, 1u << 21, false, 1) == kNone);
  // long K in a batch: rows at odd addresses, and at whole 16 bytes with the two near one another, keep 64 x 64 tiles; a single product does not
  EXPECT(plain(1956, 112, 2559, 12) == k64 && plain(896, 107, 2749, 23) == k64 && plain(773, 128, 3117, 22) == k64);
  EXPECT(plain(227, 5586, 768, 12) != kNone && plain(2752, 896, 5539) == k128);
  EXPECT(plain(704, 3656, 312) == kNone && plain(704, 3656, 320) == k128);
  // two K groups while a CU has one tile at most, but not for many tiles of a short K
  EXPECT(k_groups_of_128(1, 128) == 2 && k_groups_of_128(128, 128) == 2 && k_groups_of_128(129, 319) == 1 && k_groups_of_128(129, 320) == 2);
  EXPECT(k_groups_of_128(256, 320) == 2 && k_groups_of_128(257, 320) == 1 && k_groups_of_128(257, 8192) == 1);
  // the estimate by tiles: none where the fp32 ops have 128 x 128 tiles, otherwise no less for a k more
  EXPECT(tfcc_rocm::sgemm_tiles::microseconds(4096, 4096, 4096, 1) == 0 && tfcc_rocm::sgemm_tiles::microseconds(425, 6974, 628, 1) == 0);
  auto time = [](unsigned k) { return tfcc_rocm::sgemm_tiles::microseconds(1000, 1000, k, 1); };
  for (unsigned k = 512; k < 4096; ++k) EXPECT(time(k) > 0 && time(k + 1) >= time(k));
  // B given transposed is summed as B as stored, so the same kernel has to take it
  for (unsigned m = 48; m <= 6000; m = m * 5 / 4 + 1)
    for (unsigned n = 48; n <= 9000; n = n * 5 / 4 + 1)
      for (unsigned k = 128; k <= 9000; k = k * 4 / 3 + 1) EXPECT(plain(m, n, k) == plain(m, n, k, 1, true));
  if (failures == 0) std::printf("sgemm split plan: all passed\n");
  return failures != 0;
}
