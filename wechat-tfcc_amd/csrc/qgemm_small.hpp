// Internal interface of the quantized matmul kernel for products bound by latency (gemm_u8s8_small.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "qgemm_params.hpp"

namespace tfcc_rocm {

typedef int qgemm_v4i __attribute__((ext_vector_type(4)));

// 4x4 byte transpose: in r[q] = bytes (n0..n3) of k-row q; out c[j] = bytes (k0..k3) of column j
// v_perm_b32(hi, lo, sel): selector bytes 0-3 pick from lo, 4-7 from hi
__device__ __forceinline__ void transpose4x4(const unsigned r[4], unsigned c[4]) {
  const unsigned t0 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);  // r0.b0 r1.b0 r0.b1 r1.b1
  const unsigned t1 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);  // r0.b2 r1.b2 r0.b3 r1.b3
  const unsigned t2 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
  const unsigned t3 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
  c[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);  // t0.lo16 t2.lo16
  c[1] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);  // t0.hi16 t2.hi16
  c[2] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
  c[3] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
}

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
int qgemm_small_launch(hipStream_t stream, QGemmParams p, const QSmallOutputs& o);

}  // namespace tfcc_rocm
