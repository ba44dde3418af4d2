// Argument block shared by the fp32 GEMM kernels (register-staged in sgemm.hip, direct-to-LDS in
// sgemm_dma.hip) and the entry points that pick between them.
#pragma once

#include "common.hpp"
#include "qgemm_params.hpp"  // UDiv: division by multiply-high
#include "sgemm_skinny_plan.hpp"

namespace tfcc_rocm {
namespace sgemm_detail {

struct SgemmParams {
  const float* A;
  const float* B;
  const float* bias;
  const float* residual;  // optional, laid out like C (batch stride strideR): added after the bias
  float* C;
  unsigned long long strideA, strideB, strideC, strideR;  // between outer batch entries (elements)
  unsigned long long innerA, innerB, innerC;              // between inner batch entries
  unsigned batchInner;    // batch entry bi = (bi / batchInner, bi % batchInner); 1 for a flat batch
  unsigned lda, ldb, ldc; // row strides of A, of B (of B^T when transposed) and of C, in elements
  int act;                // 0 none, 1 erf-form GELU applied last
  // grouped form (groups > 0): batch entry g multiplies the shared A by groupB[g] into groupC[g]
  unsigned groups;
  const float* groupB[4];
  const float* groupBias[4];
  float* groupC[4];
  unsigned M, N, K, batch;
  unsigned tilesM, tilesN, tilesTotal, chunk;
  // division by tilesM * tilesN, by 4 * tilesN and by batchInner as multiply-high and shift (set_tiles)
  unsigned perBatchMagic, perBatchShift, bandMagic, bandShift, innerMagic, innerShift;
#if defined(__HIPCC__)
  __device__ __forceinline__ const SgemmParams& whole() const { return *this; }
#endif
};

// Shorter argument blocks for what most launches are: one product, a flat batch without epilogue, and (behind the leading
// scalar arguments of kernels that have those) what the tile store of one product needs.  A launch whose arguments take more than
// 112 bytes costs the host 0.65 us more in two of three processes: us from launch to launch of an empty kernel, 112 bytes 2.75,
// 116 bytes 3.4, 320 bytes 3.5 (2.3 whatever the size in the others).  A small product is bound by its launch: 1 x 768 x 768 4.42 -> 4.21 in one of them, 4.30 -> 4.23 in
// another, where runs of one side differ by as much.
// whole(): the block as the kernels read it, everything else a constant.
constexpr size_t kShortArguments = 112;

struct SgemmLone {
  const float *A, *B, *bias, *residual;
  float* C;
  unsigned lda, ldb, ldc, M, N, K, tilesM, tilesN, tilesTotal, chunk, bandMagic, bandShift;
  int act;
  explicit SgemmLone(const SgemmParams& p)
      : A(p.A), B(p.B), bias(p.bias), residual(p.residual), C(p.C), lda(p.lda), ldb(p.ldb), ldc(p.ldc), M(p.M), N(p.N), K(p.K),
        tilesM(p.tilesM), tilesN(p.tilesN), tilesTotal(p.tilesTotal), chunk(p.chunk), bandMagic(p.bandMagic), bandShift(p.bandShift),
        act(p.act) {}
  static bool takes(const SgemmParams& p) { return p.groups == 0 && p.batch == 1; }
  __device__ __forceinline__ SgemmParams whole() const {
    SgemmParams p{};
    p.A = A; p.B = B; p.bias = bias; p.residual = residual; p.C = C; p.act = act;
    p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.M = M; p.N = N; p.K = K; p.batch = p.batchInner = 1;
    p.tilesM = tilesM; p.tilesN = tilesN; p.tilesTotal = tilesTotal; p.chunk = chunk; p.bandMagic = bandMagic; p.bandShift = bandShift;
    p.perBatchShift = 31;  // with a magic number of 0: every tile is in batch entry 0
    return p;
  }
};

struct SgemmBatch {
  const float *A, *B;
  float* C;
  unsigned long long strideA, strideB, strideC;
  unsigned lda, ldb, ldc, M, N, K, tilesM, tilesN, tilesTotal, chunk, perBatchMagic, perBatchShift, bandMagic, bandShift;
  explicit SgemmBatch(const SgemmParams& p)
      : A(p.A), B(p.B), C(p.C), strideA(p.strideA), strideB(p.strideB), strideC(p.strideC), lda(p.lda), ldb(p.ldb), ldc(p.ldc), M(p.M),
        N(p.N), K(p.K), tilesM(p.tilesM), tilesN(p.tilesN), tilesTotal(p.tilesTotal), chunk(p.chunk), perBatchMagic(p.perBatchMagic),
        perBatchShift(p.perBatchShift), bandMagic(p.bandMagic), bandShift(p.bandShift) {}
  static bool takes(const SgemmParams& p) { return p.groups == 0 && p.batchInner == 1 && !p.bias && !p.residual && p.act == 0; }
  __device__ __forceinline__ SgemmParams whole() const {
    SgemmParams p{};
    p.A = A; p.B = B; p.C = C; p.strideA = strideA; p.strideB = strideB; p.strideC = strideC;
    p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.M = M; p.N = N; p.K = K; p.batchInner = 1;
    p.tilesM = tilesM; p.tilesN = tilesN; p.tilesTotal = tilesTotal; p.chunk = chunk;
    p.perBatchMagic = perBatchMagic; p.perBatchShift = perBatchShift; p.bandMagic = bandMagic; p.bandShift = bandShift;
    return p;
  }
};

struct SgemmFinish {
  const float *bias, *residual;
  float* C;
  unsigned ldc;
  int act;
  explicit SgemmFinish(const SgemmParams& p) : bias(p.bias), residual(p.residual), C(p.C), ldc(p.ldc), act(p.act) {}
  __device__ __forceinline__ SgemmParams whole() const {
    SgemmParams p{};
    p.bias = bias; p.residual = residual; p.C = C; p.ldc = ldc; p.act = act; p.batch = p.batchInner = 1;
    return p;
  }
};
static_assert(sizeof(SgemmLone) <= kShortArguments && sizeof(SgemmBatch) <= kShortArguments && sizeof(SgemmFinish) == 32, "short");

// Fills in the tile counts for BM x BN tiles; false when there are too many tiles for one grid.
inline bool set_tiles(SgemmParams& p, unsigned bm, unsigned bn) {
  p.tilesM = (p.M + bm - 1) / bm;
  p.tilesN = (p.N + bn - 1) / bn;
  const unsigned long long total = (unsigned long long)p.tilesM * p.tilesN * p.batch;
  if (total > 0x7fffffffull) return false;
  p.tilesTotal = (unsigned)total;
  p.chunk = (p.tilesTotal + 7) / 8;
  const UDiv perBatch = udiv_prepare(p.tilesM * p.tilesN), band = udiv_prepare(4u * p.tilesN),
             inner = udiv_prepare(p.batchInner);
  p.perBatchMagic = perBatch.magic; p.perBatchShift = perBatch.shift;
  p.bandMagic = band.magic; p.bandShift = band.shift;
  p.innerMagic = inner.magic; p.innerShift = inner.shift;
  return true;
}

// The direct-to-LDS kernels (sgemm_dma.hip).  `config`: 0 = 64x64 tiles, 1 = 32x96, 2 = 32x64, 3 = 32x32,
// 5 = 128x96 (serial groups only); ksplit 1 or 2 groups of wavefronts on one tile (four K groups run on the
// kernels of sgemm_wave96.hip).
// Requires B not transposed and operands below 2^30 elements.
// serialGroups: one group of wavefronts per tile does the work of the `ksplit` groups one slab after the other
// (same additions, same result) - for launches that fill the chip anyway.
int sgemm_dma_launch(hipStream_t stream, SgemmParams p, int config, int ksplit, bool serialGroups);

// The hand-scheduled kernels with one wavefront per SIMD (sgemm_wave96.hip), a wavefront owning 32 rows x `blocks`
// column blocks of 32: ksplit = 4 - tiles of 32 x 32 blocks with the four K groups as the four wavefronts of a
// workgroup (blocks 1, 2 or 3), or 64 x 64 tiles with eight wavefronts (blocks 2, rowBlocks 2); ksplit = 2 - 64 x 64 tiles (blocks 2, rowBlocks 2: two pairs of wavefronts) or 32 x 32
// (blocks 1, rowBlocks 1: two wavefronts); ksplit = 1 - tiles of 128 x 32 blocks, four wavefronts on a shared ring
// (blocks 3 or 4).  Same requirements and the same bits as the kernels above for the same number of K groups.
int sgemm_wave96_launch(hipStream_t stream, SgemmParams p, int ksplit, int blocks = 3, int rowBlocks = 0);

// The kernels on the bf16 matrix cores (sgemm_split.hip), operands split into three exact parts.  `kernel`: one of
// sgemm_split_plan.hpp.  Any alignment, B as stored or transposed (the same bits); operands
// below 2^29 elements, rows of C below 2^21.
int sgemm_split_launch(hipStream_t stream, const SgemmParams& p, int kernel, bool transB);

// The streaming kernel for up to eight rows of A (sgemv.hip): any K, N, strides and alignment; B not transposed.
bool sgemv_supported(const SgemmParams& p);
int sgemv_launch(hipStream_t stream, const SgemmParams& p);

// The kernel for few rows (sgemm_skinny.hip): one product, or the grouped form; any alignment, B as stored or transposed,
// operands below 2^30 elements.
void sgemm_skinny_release_stream(int dev, hipStream_t stream);
int sgemm_skinny_launch(hipStream_t stream, const SgemmParams& p, const sgemm_skinny_plan::Plan& plan, bool transB);

// The kernel for a K that is dealt out over the wavefronts of one or several workgroups (sgemm_deal.hip), as sgemm_deal_plan.hpp
// says: one product, or the grouped form; any alignment, B as stored or transposed, operands below 2^30 elements.
int sgemm_deal_launch(hipStream_t stream, const SgemmParams& p, unsigned splits, unsigned blocks, bool transB);
void sgemm_deal_release_stream(int dev, hipStream_t stream);

}  // namespace sgemm_detail
}  // namespace tfcc_rocm
