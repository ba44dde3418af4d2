// Which fp32 products take the kernels whose workgroups share a K (wechat-tfcc_amd/csrc/sgemm_skinny_plan.hpp), on the host: no GPU.
// With arguments, groups of m n k: prints kernel, splits and row blocks or column blocks of each product.
#include <cstdio>
#include <cstdlib>

#include "sgemm_skinny_plan.hpp"
#include "sgemm_split_plan.hpp"

using namespace tfcc_rocm;
using namespace tfcc_rocm::sgemm_skinny_plan;

static int failures = 0;
#define EXPECT(cond)                                         \
  do {                                                       \
    if (!(cond)) {                                           \
      ++failures;                                            \
      std::printf("FAIL line %d: %s\n", __LINE__, #cond);    \
    }                                                        \
  } while (0)

// of m x k times k x n, dense
static Choice chosen(unsigned m, unsigned k, unsigned n) {
  return choose(m, n, k, [&] { return sgemm_split_plan::kernel_of(m, n, k, k, n, n, false, 1) != sgemm_split_plan::kNone; });
}

int main(int argc, char** argv) {
  if (argc > 1) {
    const char* const names[] = {"other", "skinny", "deal"};
    for (int i = 1; i + 2 < argc; i += 3) {
      const Choice c = chosen(std::atoi(argv[i]), std::atoi(argv[i + 1]), std::atoi(argv[i + 2]));
      std::printf("%s %u %u\n", names[c.kernel], c.kernel == kDeal ? c.deal.splits : c.skinny.splits, c.kernel == kDeal ? c.deal.blocks : c.skinny.rows);
    }
    return 0;
  }
  for (unsigned m = 1; m <= 3000; m = m * 6 / 5 + 1)
    for (unsigned n = 1; n <= 20000; n = n * 6 / 5 + 1)
      for (unsigned k = 1; k <= 20000; k = k * 6 / 5 + 1) {
        int asked = 0;
        const Choice c = choose(m, n, k, [&] { return ++asked > 100; });
        const sgemm_deal_plan::Plan deal = sgemm_deal_plan::plan_of(m, n, k);
        EXPECT(c.deal.splits == deal.splits && c.deal.blocks == deal.blocks && c.deal.us == deal.us);
        EXPECT(asked <= (c.deal.splits > 0 && !c.skinny.better ? 1 : 0));  // the rule of the bf16 ops only where it decides
        EXPECT(c.kernel != kDeal || c.deal.splits > 0);
        // replayed, a tile of 32 x 32 has one CU: neither a second round of them nor what fills the chip without splits
        EXPECT(c.kernel != kDeal || (sgemm_deal_plan::tiles_of(m, n, 1) <= 256 && !c.skinny.unsplit));
        if (c.kernel != kSkinny) continue;
        // splits of at least 512 k, the partial tiles within the memory in which they meet
        const unsigned tall = 16 * c.skinny.rows;
        const unsigned long long tiles = (unsigned long long)((m + tall - 1) / tall) * ((n + 15) / 16);
        EXPECT(c.skinny.better && (c.skinny.rows == 1 || (c.skinny.rows == 2 && m > 16)));
        // two row blocks: one workgroup to a CU, and an XCD has a run of tiles with all their splits on 32 CUs
        if (c.skinny.rows == 2 && tiles * c.skinny.splits <= 256) EXPECT((tiles + 7) / 8 * c.skinny.splits <= 32);
        EXPECT(c.skinny.splits == 1 || (k / c.skinny.splits >= 512 && tiles * c.skinny.rows * c.skinny.splits <= kMaxParts));
      }
  // 84 tiles: eleven on an XCD, so three splits are 33 workgroups there
  EXPECT(chosen(17, 3163, 1336).skinny.rows == 1 && chosen(211, 1903, 192).skinny.rows == 1 && chosen(20, 5051, 784).skinny.rows == 1);
  // whole tiles, few columns and a K past 1024: tiled; more columns or a shorter K: two blocks
  EXPECT(chosen(960, 1120, 128).kernel == kOther && chosen(674, 1344, 144).kernel == kOther && chosen(754, 1216, 136).kernel == kOther);
  EXPECT(chosen(51, 1152, 1408).skinny.rows == 2 && chosen(618, 896, 112).skinny.rows == 2 && chosen(17, 1216, 2944).skinny.rows == 2);
  EXPECT(chosen(128, 3072, 768).kernel == kDeal && chosen(512, 6336, 456).kernel == kDeal && chosen(128, 2496, 1280).kernel == kDeal);
  EXPECT(chosen(288, 7296, 920).kernel == kOther && chosen(485, 4448, 104).kernel == kSkinny && chosen(485, 4448, 104).skinny.splits == 1);
  // whole tiles and few columns
  EXPECT(chosen(398, 1344, 208).kernel != kDeal && chosen(332, 1664, 344).kernel != kDeal && chosen(128, 1344, 768).kernel != kDeal);
  // one and two rows of whole chunks: few columns, and a B that the L2s hold, are streamed; a remainder, more rows or columns are not
  for (unsigned m = 1; m <= 2; ++m) {
    EXPECT(chosen(m, 1472, 64).kernel == kOther && chosen(m, 1216, 640).kernel == kOther && chosen(m, 2048, 3840).kernel == kOther);
    EXPECT(chosen(m, 1792, 64).kernel == kSkinny && chosen(m, 1472, 768).kernel == kSkinny && chosen(m, 1473, 64).kernel == kSkinny);
    EXPECT(chosen(m, 2304, 2304).kernel == kSkinny && chosen(m, 2048, 4096).kernel == kSkinny && chosen(m, 2048, 3841).kernel == kSkinny);
  }
  EXPECT(chosen(3, 1472, 64).kernel == kSkinny && chosen(3, 2048, 3840).kernel == kSkinny);
  if (failures == 0) std::printf("sgemm skinny plan: all passed\n");
  return failures != 0;
}
