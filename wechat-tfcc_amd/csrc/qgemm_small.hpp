// Internal interface of the quantized matmul kernel for products bound by latency (gemm_u8s8_small.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "qgemm_params.hpp"

namespace tfcc_rocm {

typedef int qgemm_v4i __attribute__((ext_vector_type(4)));

// What a load of four (sixteen) bytes that was moved back by `shift` bytes to stay inside its operand was meant to give:
// zeros behind the end.
__device__ __forceinline__ unsigned moved4(unsigned v, unsigned shift) { return shift < 4 ? v >> (8 * shift) : 0u; }
__device__ __forceinline__ qgemm_v4i moved16(qgemm_v4i v, unsigned shift) {
  unsigned w[5] = {(unsigned)v[0], (unsigned)v[1], (unsigned)v[2], (unsigned)v[3], 0u};
  if (shift & 8) { w[0] = w[2]; w[1] = w[3]; w[2] = w[3] = 0u; }
  if (shift & 4) { w[0] = w[1]; w[1] = w[2]; w[2] = w[3]; w[3] = 0u; }
  qgemm_v4i r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = shift < 16 ? (int)__builtin_amdgcn_alignbyte(w[i + 1], w[i], shift & 3) : 0;
  return r;
}

// What the kernel writes besides p.C and p.Q (either may be null): f32Out[r][n] = float(acc * scaleA * scaleB[n]).
struct QSmallOutputs {
  float* f32Out;
  const float* scaleB;
  float scaleA;
};

// Any shape and alignment; operands well below 2^31 bytes.
bool qgemm_small_supported(const QGemmParams& p);
// split: by several workgroups per tile where qgemm_small_splits says so, whether or not that beats one workgroup per tile.
int qgemm_small_launch(hipStream_t stream, QGemmParams p, const QSmallOutputs& o, bool split = false);
// Whether the product would be split over several workgroups per tile, and be faster than a kernel that takes `instead`
// hundredths of a microsecond.
bool qgemm_small_splits(hipStream_t stream, unsigned m, unsigned n, unsigned k, unsigned instead);
// Gives back what is kept for `stream` on the device (the stream must be idle).
void qgemm_small_release_stream(int dev, hipStream_t stream);

}  // namespace tfcc_rocm
