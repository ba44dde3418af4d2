// uint8 x int8 -> int32 matrix product on the gfx950 int8 matrix cores, with the offset terms of
// the reference's quantized matmul and (optionally) its requantize step fused into the tile store: the entry points and
// which kernel takes a product.
//
// Replaces tfcc/mkl/operations/tfcc_mklquantization.cpp:33-69,176-201 (offset matrix + threaded
// driver), tfcc/mkl/gemm/tfcc_mklsinglethreadgemm.h:93-141 (blocking / packing) and the 24x4x2
// micro-kernel tfcc/mkl/gemm/tfcc_mklmatmulkernel.h:142-260.
//
// A is [M,K] uint8 and B is [K,N] int8, both row-major in HBM, of any size and alignment.  The int8 product of a' = a - 128
// and b is turned into the reference's result with rank-1 terms in the epilogue of every kernel:
//   sum (a+oA)(b+oB) = sum a'b + 128*colsum(B)[j] + oB*rowsumA[i] + oA*colsumB[j] + K*oA*oB
// where rowsumA / colsumB are the caller's tensors (used as given, like the reference) and
// colsum(B) is the true column sum, accumulated on the fly from the operands so that no assumption about the caller's
// tensors is needed.
#include "common.hpp"
#include "gemv.hpp"
#include "qgemm_dma.hpp"
#include "qgemm_params.hpp"
#include "qgemm_small.hpp"

namespace tfcc_rocm {
namespace {

// Where the line lies (us; t64 is the number of 64 x 128 tiles): t64 <= 64, or at most 32 rows, go to the kernel without slabs
// (gemm_u8s8_small.hip), aligned or not - 256 x 1024 x 1024 6.2 against 8.1 in direct-to-LDS slabs, 64 x 4096 x 4096 15.5
// against 23.6, 300 x 5000 x 700 16.9 against 20; past it 512 x 1023 x 1025 17.2 against 11.5, 640 x 1024 x 1024 9.9
// against 8.3.  The rest goes to the kernels that walk K in slabs (gemm_u8s8_dma.hip).
template <bool REQUANT>
int dispatch(hipStream_t stream, const QGemmParams& p) {
  const unsigned long long t64 = (unsigned long long)((p.M + 63) / 64) * ((p.N + 127) / 128) * p.batch;
  const bool loads = (unsigned long long)p.M * p.K >= 16 && (unsigned long long)p.K * p.N >= 16;  // operands as long as one load
  if (!loads || ((t64 <= 64 || p.M <= 32) && qgemm_small_supported(p))) return qgemm_small_launch(stream, p, QSmallOutputs{});
  return qgemm_dma_launch(stream, p, REQUANT);
}

int fill_params(const tfcc_rocm_qgemm_desc* d, QGemmParams& p) {
  TFCC_REQUIRE(d != nullptr, "quantized matmul: null descriptor");
  TFCC_REQUIRE(d->a && d->b && d->rowsum_a && d->colsum_b, "quantized matmul: null operand");
  TFCC_REQUIRE(d->m > 0 && d->n > 0 && d->k > 0 && d->batch > 0, "quantized matmul: empty operand");
  const bool anyRange = d->min_a || d->max_a || d->min_b || d->max_b;
  const bool allRange = d->min_a && d->max_a && d->min_b && d->max_b;
  TFCC_REQUIRE(!anyRange || allRange, "quantized matmul: give all four range pointers or none");
  TFCC_REQUIRE((unsigned long long)d->m * d->n < (1ull << 32) && (unsigned long long)d->m * d->k < (1ull << 32) &&
               ((unsigned long long)d->k + 256) * d->n + 512 < (1ull << 32),
               "quantized matmul: operand larger than 2^32 elements");
  p = QGemmParams{};
  p.A = d->a; p.B = d->b; p.rowsumA = d->rowsum_a; p.colsumB = d->colsum_b;
  p.strideA = d->stride_a; p.strideB = d->stride_b; p.strideRA = d->stride_rowsum_a;
  p.strideRB = d->stride_colsum_b; p.strideC = d->stride_c;
  p.M = d->m; p.N = d->n; p.K = d->k; p.batch = d->batch;
  p.offsetA = d->offset_a; p.offsetB = d->offset_b;
  p.colsumExact = d->colsum_b_is_exact ? 1 : 0;
  if (allRange) { p.minA = d->min_a; p.maxA = d->max_a; p.minB = d->min_b; p.maxB = d->max_b; p.minC = d->min_c; p.maxC = d->max_c; }
  return TFCC_ROCM_OK;
}

}  // namespace
}  // namespace tfcc_rocm

using namespace tfcc_rocm;

extern "C" int tfcc_rocm_gemm_u8s8s32(void* stream, const tfcc_rocm_qgemm_desc* desc, int32_t* c) {
  QGemmParams p;
  if (int e = fill_params(desc, p)) return e;
  TFCC_REQUIRE(c != nullptr, "quantized matmul: null result");
  p.C = c;
  // decode shapes: a few rows against a large B are bandwidth bound and take the skinny kernel, on the
  // packed copy of B when the caller has one
  if (desc->packed_b && p.batch == 1 && gemv_packed_supported(p.A, desc->packed_b, p.M, p.K)) {
    const float* ranges[4] = {p.minA, p.maxA, p.minB, p.maxB};
    float* rangeOut[2] = {p.minC, p.maxC};
    return gemv_packed_launch(as_stream(stream), p.A, desc->packed_b, p.rowsumA, p.colsumB, p.offsetA, p.offsetB,
                              ranges, rangeOut, p.M, p.N, p.K, c, 0.f, nullptr, nullptr);
  }
  if (p.batch == 1 && p.M <= 8 && (unsigned long long)p.N * p.K >= (1u << 20) &&
      (gemv_supported(p.A, p.B, p.M, p.N, p.K) || gemv_wide_takes_ragged(p.M, p.N, p.K, p.colsumExact != 0))) {
    const float* ranges[4] = {p.minA, p.maxA, p.minB, p.maxB};
    float* rangeOut[2] = {p.minC, p.maxC};
    return gemv_launch(as_stream(stream), p.A, p.B, p.rowsumA, p.colsumB, p.offsetA, p.offsetB, ranges, rangeOut,
                       p.M, p.N, p.K, c, 0.f, nullptr, nullptr, p.colsumExact != 0);
  }
  return dispatch<false>(as_stream(stream), p);
}

extern "C" int tfcc_rocm_gemm_u8s8s32_requant_u8(void* stream, const tfcc_rocm_qgemm_desc* desc,
                                                 int32_t* acc_out, uint8_t* q_out, double in_scale,
                                                 double in_min, double out_scale, int64_t out_offset,
                                                 const float* min_out, const float* max_out) {
  QGemmParams p;
  if (int e = fill_params(desc, p)) return e;
  TFCC_REQUIRE(q_out != nullptr, "quantized matmul: null requantized result");
  TFCC_REQUIRE((min_out == nullptr) == (max_out == nullptr), "quantized matmul: give both output range pointers or none");
  TFCC_REQUIRE(min_out == nullptr || p.minA != nullptr,
               "quantized matmul: an output range in device memory needs the operand ranges in the descriptor");
  p.C = acc_out;
  p.Q = q_out;
  p.inScale = in_scale; p.inMin = in_min; p.outScale = out_scale; p.outOffset = out_offset;
  p.minOut = min_out; p.maxOut = max_out;
  return dispatch<true>(as_stream(stream), p);
}
