// Bandwidth-bound companions of the quantized matmul: int32 row / column sums, and the
// range-based quantize / requantize / dequantize steps with their scale arithmetic evaluated on
// the device in double (the ranges are float scalars in device memory, as the reference passes
// them as tensors).
//
// Replaces tfcc/mkl/operations/tfcc_mklquantization.cpp:205-318 (reduce_sum),
// tfcc/mkl/kernel/tfcc_mklquantizationkernel.avx256.cpp:55-145 (the AVX2 kernels: nearest-even
// rounding, fused multiply-add) and the branches of
// tfcc/mkl/interfaces/tfcc_mklquantizationinterface.cpp:47-69,72-147,191-240,284-333.
#include <atomic>

#include "common.hpp"
#include "quant_ops.hpp"
#include "quantize_exchange.hpp"
#include "stream_slots.hpp"

namespace tfcc_rocm {
namespace {

template <class T>
__device__ __forceinline__ long long load_as_i64(const void* p, size_t i) {
  return (long long)static_cast<const T*>(p)[i];
}

__device__ __forceinline__ long long load_typed(const void* p, int type, size_t i) {
  switch (type) {
    case TFCC_ROCM_S8: return load_as_i64<int8_t>(p, i);
    case TFCC_ROCM_U8: return load_as_i64<uint8_t>(p, i);
    case TFCC_ROCM_S16: return load_as_i64<int16_t>(p, i);
    case TFCC_ROCM_U16: return load_as_i64<uint16_t>(p, i);
    case TFCC_ROCM_S32: return load_as_i64<int32_t>(p, i);
    default: return load_as_i64<uint32_t>(p, i);
  }
}

__device__ __forceinline__ void store_typed(void* p, int type, size_t i, long long v) {
  switch (type) {
    case TFCC_ROCM_S8: static_cast<int8_t*>(p)[i] = (int8_t)v; break;
    case TFCC_ROCM_U8: static_cast<uint8_t*>(p)[i] = (uint8_t)v; break;
    case TFCC_ROCM_S16: static_cast<int16_t*>(p)[i] = (int16_t)v; break;
    case TFCC_ROCM_U16: static_cast<uint16_t*>(p)[i] = (uint16_t)v; break;
    case TFCC_ROCM_S32: static_cast<int32_t*>(p)[i] = (int32_t)v; break;
    default: static_cast<uint32_t*>(p)[i] = (uint32_t)v; break;
  }
}

// ---- row sums: one wavefront per row, 16-byte loads at any address (rows of an odd length start anywhere).  Bound by
// the launch and one trip to memory.
template <class T>
__global__ __launch_bounds__(256) void reduce_rows_kernel(const T* a, unsigned rows, unsigned col, int* out) {
  const unsigned wave = (blockIdx.x * 256 + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  if (wave >= rows) return;
  const T* p = a + (size_t)wave * col;
  unsigned s = 0;
  constexpr unsigned PER = 16 / sizeof(T);
  const unsigned chunks = col / PER, rest = col - chunks * PER;
  // the elements behind the last whole piece, asked for with the pieces: lanes behind them add zero
  const T tail = lane < rest ? p[chunks * PER + lane] : T(0);
  // eight loads in flight per lane; bytes are summed four at a time by the dot-product instructions
  for (unsigned i0 = lane; i0 < chunks; i0 += 64 * 8) {
    uint4 q[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      q[u] = make_uint4(0, 0, 0, 0);
      if (i0 + 64 * u < chunks) __builtin_memcpy(&q[u], p + (size_t)(i0 + 64 * u) * PER, 16);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const unsigned w[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        if (sizeof(T) == 1) {
          if (T(-1) < T(0)) s = (unsigned)__builtin_amdgcn_sdot4((int)w[d], 0x01010101, (int)s, false);
          else s = __builtin_amdgcn_udot4(w[d], 0x01010101u, s, false);
        } else {
#pragma unroll
          for (int b = 0; b < 2; ++b) s += (unsigned)(int)(T)(w[d] >> (16 * b));
        }
      }
    }
  }
  s += (unsigned)(int)tail;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (lane == 0) out[wave] = (int)s;
}

// ---- column sums: a workgroup owns 256 x (4 bytes) columns of one batch entry and a slab of rows;
// slabs are combined with integer atomics (exact and order independent) into a zeroed result.
template <class T>
__global__ __launch_bounds__(256) void reduce_cols_kernel(const T* a, unsigned row, unsigned col,
                                                          unsigned rowsPerSlab, int* out) {
  const unsigned b = blockIdx.z;
  const unsigned c = blockIdx.x * 256 + threadIdx.x;
  const unsigned r0 = blockIdx.y * rowsPerSlab;
  const unsigned r1 = min(r0 + rowsPerSlab, row);
  if (c >= col) return;
  const T* p = a + (size_t)b * row * col + c;
  unsigned s = 0;
  for (unsigned r = r0; r < r1; ++r) s += (unsigned)(int)p[(size_t)r * col];
  atomicAdd(reinterpret_cast<unsigned*>(out) + (size_t)b * col + c, s);
}

template <class T>
__global__ __launch_bounds__(256) void reduce_cols_vec_kernel(const T* a, unsigned row, unsigned col,
                                                              unsigned rowsPerSlab, int* out) {
  // col % 4 == 0 and 4-byte aligned rows (1-byte types): one dword = 4 columns per thread
  const unsigned b = blockIdx.z;
  const unsigned c4 = blockIdx.x * 256 + threadIdx.x;
  const unsigned r0 = blockIdx.y * rowsPerSlab;
  const unsigned r1 = min(r0 + rowsPerSlab, row);
  if (c4 * 4 >= col) return;
  const unsigned* p = reinterpret_cast<const unsigned*>(a + (size_t)b * row * col) + c4;
  const unsigned pitch = col / 4;
  unsigned s[4] = {0, 0, 0, 0};
  for (unsigned r = r0; r < r1; ++r) {
    unsigned w = p[(size_t)r * pitch];
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += (unsigned)(int)(T)(w >> (8 * e));
  }
  unsigned* o = reinterpret_cast<unsigned*>(out) + (size_t)b * col + c4 * 4;
#pragma unroll
  for (int e = 0; e < 4; ++e) atomicAdd(o + e, s[e]);
}

// 16-byte loads of data that is read once
typedef int nt_v4i __attribute__((ext_vector_type(4)));
typedef float nt_v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int4 load_streamed(const int4* p) {
  const nt_v4i v = __builtin_nontemporal_load(reinterpret_cast<const nt_v4i*>(p));
  return make_int4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ float4 load_streamed(const float4* p) {
  const nt_v4f v = __builtin_nontemporal_load(reinterpret_cast<const nt_v4f*>(p));
  return make_float4(v[0], v[1], v[2], v[3]);
}

// Column sums of a 1-byte type with col % 16 == 0 and 16-byte aligned rows.  A workgroup owns 1024 columns
// (64 threads x 16 bytes: whole 1 KB row segments) and a slab of rows, dealt to four row lanes.  A thread takes its
// rows four at a time, transposes each 4 x 4 byte block in registers so that a word holds one column's four rows,
// and adds those with one dot-product instruction; the four row lanes meet in LDS and the slab's sums go to the
// (zeroed) result with integer atomics, whose order does not matter.
template <class T>
__global__ __launch_bounds__(256) void reduce_cols_wide_kernel(const T* a, unsigned row, unsigned col,
                                                               unsigned rowsPerSlab, int* out) {
  constexpr bool kSigned = T(-1) < T(0);
  __shared__ int part[4][64][17];
  const unsigned b = blockIdx.z, cg = threadIdx.x & 63u, rl = threadIdx.x >> 6;
  const unsigned c16 = blockIdx.x * 64 + cg;
  const unsigned r0 = blockIdx.y * rowsPerSlab, r1 = min(r0 + rowsPerSlab, row);
  int s[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) s[e] = 0;
  if (c16 * 16 < col) {
    const size_t pitch = col / 16;
    const int4* p = reinterpret_cast<const int4*>(a + (size_t)b * row * col) + c16;
    unsigned r = r0 + rl;
#pragma unroll 2
    for (; r + 12 < r1; r += 16) {
      const int4 v0 = load_streamed(p + (size_t)r * pitch), v1 = load_streamed(p + (size_t)(r + 4) * pitch),
                 v2 = load_streamed(p + (size_t)(r + 8) * pitch), v3 = load_streamed(p + (size_t)(r + 12) * pitch);
      const unsigned w[4][4] = {{(unsigned)v0.x, (unsigned)v1.x, (unsigned)v2.x, (unsigned)v3.x},
                                {(unsigned)v0.y, (unsigned)v1.y, (unsigned)v2.y, (unsigned)v3.y},
                                {(unsigned)v0.z, (unsigned)v1.z, (unsigned)v2.z, (unsigned)v3.z},
                                {(unsigned)v0.w, (unsigned)v1.w, (unsigned)v2.w, (unsigned)v3.w}};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        unsigned c[4];
        transpose4x4(w[d], c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          s[4 * d + e] = kSigned ? __builtin_amdgcn_sdot4((int)c[e], 0x01010101, s[4 * d + e], false)
                                 : (int)__builtin_amdgcn_udot4(c[e], 0x01010101u, (unsigned)s[4 * d + e], false);
      }
    }
    for (; r < r1; r += 4) {
      const int4 v = load_streamed(p + (size_t)r * pitch);
      const unsigned w[4] = {(unsigned)v.x, (unsigned)v.y, (unsigned)v.z, (unsigned)v.w};
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[4 * d + e] += (int)(T)(w[d] >> (8 * e));
    }
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) part[rl][cg][e] = s[e];
  __syncthreads();
  // 1024 sums per workgroup, four per thread
  unsigned* o = reinterpret_cast<unsigned*>(out) + (size_t)b * col;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const unsigned idx = threadIdx.x + 256u * q, g = idx >> 4, e = idx & 15u;
    const unsigned column = (blockIdx.x * 64 + g) * 16 + e;
    if (column < col) atomicAdd(o + column, (unsigned)(part[0][g][e] + part[1][g][e] + part[2][g][e] + part[3][g][e]));
  }
}

__global__ void zero_kernel(int* p, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---- requantize / dequantize / quantize -----------------------------------------------------
__global__ __launch_bounds__(256) void requantize_kernel(const void* in, int inType, void* out, int outType,
                                                         size_t total, const float* minIn, const float* maxIn,
                                                         const float* minOut, const float* maxOut) {
  const RequantScalars s = make_requant_scalars(inType, outType, *minIn, *maxIn, *minOut, *maxOut);
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (; i < total; i += step) {
    long long q = s.fillValue;
    if (!s.mode) {
      const long long x = load_typed(in, inType, i);
      q = s.fastOK ? (long long)requantize_one_fast((double)(x - s.inLowest), s) : requantize_one_exact(x, s);
    }
    store_typed(out, outType, i, q);
  }
}


// int32 -> uint8, the matmul epilogue's type pair.  Four elements per 16-byte load, four loads in flight per
// thread, few enough threads that the scalar set-up (a few hundred double operations) is not what the launch
// spends its time on.
template <int FLAVOUR>  // 1 double shortcut, 2 exact int64, 3 fill, 4 int32 shortcut, 5 folded
__device__ __forceinline__ unsigned requantize_four(const int4& v, const RequantScalars& s) {
  const int x[4] = {v.x, v.y, v.z, v.w};
  unsigned q[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const double off = (double)((unsigned)x[e] ^ 0x80000000u);
    if (FLAVOUR == 5) q[e] = (unsigned)requantize_one_folded(off, s);
    else if (FLAVOUR == 4) q[e] = (unsigned)requantize_one_fast32(off, s);
    else if (FLAVOUR == 1) q[e] = (unsigned)requantize_one_fast(off, s);
    else if (FLAVOUR == 2) q[e] = (unsigned)requantize_one_exact(x[e], s);
    else q[e] = (unsigned)s.fillValue;
  }
  return (q[0] | (q[1] << 8)) | ((q[2] | (q[3] << 8)) << 16);
}

template <int FLAVOUR>
__device__ __forceinline__ void requantize_s32_u8_loop(const int4* in, unsigned* out, size_t total4, const RequantScalars& s) {
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total4; i += 4 * step) {
    int4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u * step < total4) v[u] = load_streamed(in + i + u * step);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u * step < total4) out[i + u * step] = requantize_four<FLAVOUR>(v[u], s);
  }
}

__global__ __launch_bounds__(256) void requantize_s32_u8_vec_kernel(const int4* in, unsigned* out, size_t total4,
                                                                    const float* minIn, const float* maxIn,
                                                                    const float* minOut, const float* maxOut) {
  const RequantScalars s = make_requant_scalars(TFCC_ROCM_S32, TFCC_ROCM_U8, *minIn, *maxIn, *minOut, *maxOut);
  if (s.mode) requantize_s32_u8_loop<3>(in, out, total4, s);
  else if (s.foldedOK) requantize_s32_u8_loop<5>(in, out, total4, s);
  else if (s.fast32OK) requantize_s32_u8_loop<4>(in, out, total4, s);
  else if (s.fastOK) requantize_s32_u8_loop<1>(in, out, total4, s);
  else requantize_s32_u8_loop<2>(in, out, total4, s);
}

// int32 -> float, four elements per thread and load (the accumulators of a quantized matmul)
__global__ __launch_bounds__(256) void dequantize_s32_vec_kernel(const int4* in, size_t total, const float* minV,
                                                                 const float* maxV, float4* out) {
  const size_t total4 = total / 4;
  const float mn = *minV, mx = *maxV;
  double scale = 0, minRounded = 0;
  const bool constant = mn >= mx;  // tfcc_mklquantizationinterface.cpp:321-324
  if (!constant) dequantized_scale_info(32, mn, mx, &scale, &minRounded);
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total4; i += 4 * step) {
    int4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u * step < total4) v[u] = load_streamed(in + i + u * step);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i + u * step >= total4) continue;
      float4 r = make_float4(mn, mn, mn, mn);
      if (!constant) {
        // (double)x - (double)INT32_MIN, exact in double
        r.x = (float)fma((double)((unsigned)v[u].x ^ 0x80000000u), scale, minRounded);
        r.y = (float)fma((double)((unsigned)v[u].y ^ 0x80000000u), scale, minRounded);
        r.z = (float)fma((double)((unsigned)v[u].z ^ 0x80000000u), scale, minRounded);
        r.w = (float)fma((double)((unsigned)v[u].w ^ 0x80000000u), scale, minRounded);
      }
      out[i + u * step] = r;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < (unsigned)(total & 3)) {  // the last 1..3 elements
    const size_t i = total4 * 4 + threadIdx.x;
    const unsigned x = (unsigned)reinterpret_cast<const int*>(in)[i];
    reinterpret_cast<float*>(out)[i] = constant ? mn : (float)fma((double)(x ^ 0x80000000u), scale, minRounded);
  }
}

__global__ __launch_bounds__(256) void dequantize_kernel(const void* in, int inType, size_t total,
                                                         const float* minV, const float* maxV, float* out) {
  const float mn = *minV, mx = *maxV;
  const IntRange r = int_range(inType);
  double scale = 0, minRounded = 0;
  const bool constant = mn >= mx;  // tfcc_mklquantizationinterface.cpp:321-324
  if (!constant) dequantized_scale_info(r.bits, mn, mx, &scale, &minRounded);
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (; i < total; i += step) {
    if (constant) {
      out[i] = mn;
    } else {
      double off = (double)load_typed(in, inType, i) - (double)r.lowest;
      out[i] = (float)fma(off, scale, minRounded);
    }
  }
}

__device__ __forceinline__ long long quantize_one(float x, double scale, long long offset, const IntRange& r) {
  long long q = to_int64_x86(rint((double)x * scale));
  q = (long long)((unsigned long long)q - (unsigned long long)offset + (unsigned long long)r.lowest);
  q = q < r.lowest ? r.lowest : q;
  return q > r.highest ? r.highest : q;
}

// quantize_one for values between mn and mx, or NaN: 32-bit whole numbers where all of them fit, half the instructions.
struct QuantizeScalars {
  double scale;
  long long offset;
  IntRange r;
  bool fill, narrow;
  int shift, nan;  // narrow: lowest - offset, and what a NaN becomes
};
__device__ __forceinline__ QuantizeScalars make_quantize_scalars(int outType, float mn, float mx) {
  QuantizeScalars s;
  s.r = int_range(outType);
  s.fill = mn == mx;  // tfcc_mklquantizationinterface.cpp:58-61
  s.scale = 0;
  s.offset = 0;
  if (!s.fill) quantized_scale_info(s.r.bits, mn, mx, &s.scale, &s.offset);
  s.narrow = !s.fill && s.r.bits <= 16 && fabs((double)mn * s.scale) < 0x1p29 && fabs((double)mx * s.scale) < 0x1p29;
  s.shift = (int)(s.r.lowest - s.offset);
  s.nan = s.narrow ? (int)quantize_one(__builtin_nanf(""), s.scale, s.offset, s.r) : 0;
  return s;
}
__device__ __forceinline__ long long quantize_one(float x, const QuantizeScalars& s) {
  if (s.fill) return s.r.lowest;
  if (!s.narrow) return quantize_one(x, s.scale, s.offset, s.r);
  const int q = (int)rint((double)x * s.scale) + s.shift;
  return x != x ? s.nan : min(max(q, (int)s.r.lowest), (int)s.r.highest);
}

__global__ __launch_bounds__(256) void quantize_kernel(const float* in, size_t total, const float* minV,
                                                       const float* maxV, void* out, int outType, int fromData) {
  const float mn = *minV, mx = *maxV;
  const IntRange r = int_range(outType);
  // given range: min >= max fills with lowest (tfcc_mklquantizationinterface.cpp:229-232);
  // range taken from the data: min == max fills with lowest (:58-61)
  const bool fillLowest = fromData ? (mn == mx) : (mn >= mx);
  double scale = 0;
  long long offset = 0;
  if (!fillLowest) quantized_scale_info(r.bits, mn, mx, &scale, &offset);
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (; i < total; i += step) {
    long long q = r.lowest;
    if (!fillLowest) q = quantize_one(in[i], scale, offset, r);
    store_typed(out, outType, i, q);
  }
}

// float -> uint8 / int8, four elements per thread and load, four loads in flight
__global__ __launch_bounds__(256) void quantize_8bit_vec_kernel(const float4* in, size_t total, const float* minV,
                                                                const float* maxV, unsigned* out, int outType,
                                                                int fromData) {
  const size_t total4 = total / 4;
  const float mn = *minV, mx = *maxV;
  const IntRange r = int_range(outType);
  const bool fillLowest = fromData ? (mn == mx) : (mn >= mx);
  double scale = 0;
  long long offset = 0;
  if (!fillLowest) quantized_scale_info(r.bits, mn, mx, &scale, &offset);
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total4; i += 4 * step) {
    float4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u * step < total4) v[u] = load_streamed(in + i + u * step);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i + u * step >= total4) continue;
      const float x[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
      unsigned word = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const long long q = fillLowest ? r.lowest : quantize_one(x[e], scale, offset, r);
        word |= ((unsigned)q & 0xffu) << (8 * e);
      }
      out[i + u * step] = word;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < (unsigned)(total & 3)) {  // the last 1..3 elements
    const size_t i = total4 * 4 + threadIdx.x;
    const float x = reinterpret_cast<const float*>(in)[i];
    store_typed(out, outType, i, fillLowest ? r.lowest : quantize_one(x, scale, offset, r));
  }
}

// min / max of a float tensor.  Monotone uint encoding so that unsigned atomics order floats.
__device__ __forceinline__ unsigned enc(float f) {
  unsigned u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float dec(unsigned u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// A small tensor in one launch: every workgroup reads all of it for the range, which every one of them finds alike, and
// quantizes 4096 elements.  Bound by that read: the caches deliver about 64 bytes per clock to a CU, against three or
// four launches.
constexpr unsigned kWholeLimit = 128 * 1024;  // elements; 4096 elements: 18.6 -> 3.4 us per call, 77077: 6.3, 131072: 7.7 against
// 8.6 for the form in two launches, whose time does not grow with the size there
constexpr unsigned kWholeBest = 40 * 1024;  // up to where the form below is no faster: 16384 elements 3.9 us here and 4.5 there, 32768
// 4.4 (4.7 from memory) and 4.5; there the host has to ask, in 0.2 us, whether the stream is being captured
__global__ __launch_bounds__(1024) void quantize_whole_kernel(const float* in, unsigned total, void* out, int outType,
                                                              float* mnOut, float* mxOut) {
  __shared__ float shMn[16], shMx[16];
  const unsigned total4 = total / 4, rest = total & 3u, own = blockIdx.x * 1024 + threadIdx.x;
  float mine[4] = {0.f, 0.f, 0.f, 0.f};
  const unsigned count = own < total4 ? 4u : own == total4 ? rest : 0u;  // elements this thread quantizes
  if (count == 4) {
    __builtin_memcpy(mine, in + (size_t)own * 4, 16);
  } else {
#pragma unroll
    for (unsigned e = 0; e < 3; ++e)
      if (e < count) mine[e] = in[(size_t)own * 4 + e];
  }
  float mn = 3.402823466e+38f, mx = -3.402823466e+38f;
  if (threadIdx.x < rest) mn = mx = in[(size_t)total4 * 4 + threadIdx.x];
  mn = fminf(mn, 3.402823466e+38f);
  mx = fmaxf(mx, -3.402823466e+38f);
  for (unsigned i = threadIdx.x; i < total4; i += 8 * 1024) {
    float v[8][4];
#pragma unroll
    for (unsigned u = 0; u < 8; ++u)
      if (i + u * 1024 < total4) __builtin_memcpy(v[u], in + (size_t)(i + u * 1024) * 4, 16);
#pragma unroll
    for (unsigned u = 0; u < 8; ++u) {
      if (i + u * 1024 >= total4) continue;
      mn = fminf(fminf(mn, fminf(v[u][0], v[u][1])), fminf(v[u][2], v[u][3]));
      mx = fmaxf(fmaxf(mx, fmaxf(v[u][0], v[u][1])), fmaxf(v[u][2], v[u][3]));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, off, 64));
    mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    shMn[threadIdx.x >> 6] = mn;
    shMx[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    mn = fminf(mn, shMn[w]);
    mx = fmaxf(mx, shMx[w]);
  }
  if (own == 0) {
    *mnOut = mn;
    *mxOut = mx;
  }
  if (count == 0) return;
  const QuantizeScalars scalars = make_quantize_scalars(outType, mn, mx);
  long long q[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) q[e] = quantize_one(mine[e], scalars);
  if (count == 4 && scalars.r.bits == 8 && ((uintptr_t)out & 3u) == 0) {
    unsigned word = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) word |= ((unsigned)q[e] & 0xffu) << (8 * e);
    static_cast<unsigned*>(out)[own] = word;
    return;
  }
#pragma unroll
  for (unsigned e = 0; e < 4; ++e)
    if (e < count) store_typed(out, outType, (size_t)own * 4 + e, q[e]);
}

// The running minimum / maximum live, order-encoded as unsigned words, in the caller's own result words
// until the finish kernel decodes them in place: no scratch memory that calls on other streams could share.
__global__ void minmax_init_kernel(unsigned* mnWord, unsigned* mxWord) {
  *mnWord = 0xffffffffu;
  *mxWord = 0u;
}

__global__ __launch_bounds__(256) void minmax_kernel(const float* in, size_t total, unsigned* mnWord,
                                                     unsigned* mxWord) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  float mn = 3.402823466e+38f, mx = -3.402823466e+38f;
  for (; i < total; i += step) {
    float v = in[i];
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mn = fminf(mn, __shfl_down(mn, off, 64));
    mx = fmaxf(mx, __shfl_down(mx, off, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    atomicMin(mnWord, enc(mn));
    atomicMax(mxWord, enc(mx));
  }
}

// The same reduction without atomics on the result, in one launch: every workgroup leaves its minimum and maximum in the
// (not yet written) output buffer of the quantize call, and the workgroup that arrives last reduces those.  65536 atomics
// on two words took 380 us for 16.7 M floats; this takes the time of reading them once.  A launch more for the last step
// cost 3.7 us of the host's time and 1.8 us on the device; a call that may not count on a word of its stream's (a graph
// being recorded) makes it (131073 elements 7.1 us in a replay, 16.7 M 33; with the atomics 15 and 400).
constexpr unsigned kArrivalSlots = 1024, kArrivalPitch = 16;
__device__ unsigned arrivals[kArrivalSlots * kArrivalPitch];  // zero between launches: the last workgroup sees to it

template <int WAVES, bool COUNTED>
__global__ __launch_bounds__(64 * WAVES) void minmax_partial_kernel(const float* in, size_t total, float* partials,
                                                                    unsigned slot, float* mnOut, float* mxOut) {
  __shared__ float shMn[WAVES], shMx[WAVES];
  __shared__ unsigned last;
  const size_t total4 = total / 4, step = (size_t)gridDim.x * blockDim.x;
  const float4* in4 = reinterpret_cast<const float4*>(in);
  float mn = 3.402823466e+38f, mx = -3.402823466e+38f;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total4; i += 4 * step) {
    float4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u * step < total4) v[u] = load_streamed(in4 + i + u * step);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i + u * step >= total4) continue;
      mn = fminf(fminf(mn, fminf(v[u].x, v[u].y)), fminf(v[u].z, v[u].w));
      mx = fmaxf(fmaxf(mx, fmaxf(v[u].x, v[u].y)), fmaxf(v[u].z, v[u].w));
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < total - total4 * 4) {  // the last 1..3 elements
    const float v = in[total4 * 4 + threadIdx.x];
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  auto join = [&]() {  // the workgroup's minimum and maximum
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      mn = fminf(mn, __shfl_down(mn, off, 64));
      mx = fmaxf(mx, __shfl_down(mx, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
      shMn[threadIdx.x >> 6] = mn;
      shMx[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      mn = fminf(mn, shMn[w]);
      mx = fmaxf(mx, shMx[w]);
    }
  };
  join();
  if constexpr (!COUNTED) {
    if (threadIdx.x == 0) {
      partials[2 * blockIdx.x] = mn;
      partials[2 * blockIdx.x + 1] = mx;
    }
    return;
  }
  if (threadIdx.x == 0) {
    __hip_atomic_store(partials + 2 * blockIdx.x, mn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(partials + 2 * blockIdx.x + 1, mx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // Both stores go past the caches by themselves, so waiting for them is all the order there has to be: a release
    // would write back whatever the kernel before has left in this L2 (7.1 us with it, 5.6 without).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(arrivals + slot * kArrivalPitch, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return;
  for (unsigned i = threadIdx.x; i < gridDim.x; i += 64 * WAVES) {
    mn = fminf(mn, __hip_atomic_load(partials + 2 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    mx = fmaxf(mx, __hip_atomic_load(partials + 2 * i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  }
  join();
  if (threadIdx.x == 0) {
    *mnOut = mn;
    *mxOut = mx;
    __hip_atomic_store(arrivals + slot * kArrivalPitch, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The last step as a launch of its own.
__global__ __launch_bounds__(256) void minmax_final_kernel(const float* partials, unsigned blocks, float* mnOut, float* mxOut) {
  __shared__ float shMn[4], shMx[4];
  float mn = 3.402823466e+38f, mx = -3.402823466e+38f;
  for (unsigned i = threadIdx.x; i < blocks; i += 256) {
    mn = fminf(mn, partials[2 * i]);
    mx = fmaxf(mx, partials[2 * i + 1]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    mn = fminf(mn, __shfl_down(mn, off, 64));
    mx = fmaxf(mx, __shfl_down(mx, off, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    shMn[threadIdx.x >> 6] = mn;
    shMx[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    *mnOut = fminf(fminf(shMn[0], shMn[1]), fminf(shMn[2], shMn[3]));
    *mxOut = fmaxf(fmaxf(shMx[0], shMx[1]), fmaxf(shMx[2], shMx[3]));
  }
}

__global__ void minmax_finish_kernel(float* mn, float* mx) {
  *mn = dec(*reinterpret_cast<const unsigned*>(mn));
  *mx = dec(*reinterpret_cast<const unsigned*>(mx));
}

// A tensor that the GPU's registers hold, in one launch: a workgroup reads its part once, the workgroups tell one another its
// minimum and maximum, and each quantizes what it has.  A word of the exchange is half a value and the number of the call
// (quantize_exchange.hpp), so a reader waits for this call's, and nothing has to be cleared or ordered.  Calls take turns with
// kTogetherTurns sets of words.
//
// Workgroups that find no room on the GPU beside other work, and words that another call in the same set, on another stream, has
// overwritten, are not waited for: a workgroup that has waited `waitTicks` reads a part that is missing itself and tells
// the others, each another one as far as there are as many, until nothing is missing.  So nobody needs anybody, every round
// of that has one part less to look for, and the input is read about twice, as with a launch for the range.  (A replayed graph would
// find the words of its last replay, so a recorded call takes the launches below; so do large calls from several streams.)
//
// Bound by the launch, a store to memory and a load from it; with many elements to a workgroup by the reading.  us, the range
// and the quantizing in a launch each before (up to 131072 elements the form above), input from memory: 77077 7.3 -> 5.4, 131072
// 9.0 -> 5.4, 786432 8.8 -> 6.8, 2 M 11.3 -> 8.9, 8 M 21.0 -> 16.9.  (A workgroup's words stored one after the other by one thread: 7.8,
// 9.9, 17.9 from 786432 on, and 7.9, 10.4, 18.4 with a load for each as well; minima and maxima in arrays of their own 7.3, 9.3, 17.4.)
// 8 M elements beside 8192 x 4096 x 8192 products on another stream, whose workgroups leave room as they end: 358 us with a launch for
// the range, 369 here, and 3300 where a workgroup that had waited read all of the input itself.
constexpr unsigned kTogetherWorkgroups = quantize_exchange::kWorkgroups, kTogetherTurns = 256;
constexpr unsigned kTogetherWait = 10;  // us (8 M elements beside other work: 366 us with 5, 369 with 10, 376 with 20, 402 with 50, 549 with 200; alone 5
// are enough and 2 too few: 25 instead of 14 in cache)
__device__ __attribute__((aligned(64))) unsigned long long togetherWords[kTogetherTurns * kTogetherWorkgroups * quantize_exchange::kWords];

typedef unsigned together_v4u __attribute__((ext_vector_type(4)));
constexpr int kDeviceScope = 16;  // sc1, as a load of an atomic at device scope has it

template <int QUADS>
__global__ __launch_bounds__(1024) void quantize_together_kernel(const float* in, size_t total, void* out, int outType, float* mnOut,
                                                                 float* mxOut, unsigned long long number, unsigned long long waitTicks) {
  namespace exchange = quantize_exchange;
  constexpr float kNoMinimum = 3.402823466e+38f, kNoMaximum = -3.402823466e+38f;
  __shared__ float shMn[16], shMx[16];
  __shared__ unsigned long long shMissing[kTogetherWorkgroups / 64];
  const size_t total4 = total / 4, first = (size_t)blockIdx.x * (1024 * QUADS) + threadIdx.x;
  const unsigned rest = (unsigned)(total & 3u);
  auto read = [&](float (&v)[4], size_t i) __attribute__((always_inline)) {  // NaN behind the end, which a range passes over
    if (i < total4) __builtin_memcpy(v, in + i * 4, 16);
    else
#pragma unroll
      for (unsigned e = 0; e < 4; ++e) v[e] = i == total4 && e < rest ? in[i * 4 + e] : __builtin_nanf("");
  };
  auto widen = [](float& low, float& high, const float (&v)[4]) __attribute__((always_inline)) {
    low = fminf(fminf(low, fminf(v[0], v[1])), fminf(v[2], v[3]));
    high = fmaxf(fmaxf(high, fmaxf(v[0], v[1])), fmaxf(v[2], v[3]));
  };
  auto join = [&](float& low, float& high, auto&& beside) __attribute__((always_inline)) {  // over the workgroup
    low = wave_min(low);
    high = wave_max(high);
    __syncthreads();  // the last join's values are read
    if ((threadIdx.x & 63) == 0) {
      shMn[threadIdx.x >> 6] = low;
      shMx[threadIdx.x >> 6] = high;
      beside();
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      low = fminf(low, shMn[w]);
      high = fmaxf(high, shMx[w]);
    }
  };
  float v[QUADS][4], mn = kNoMinimum, mx = kNoMaximum;
#pragma unroll
  for (int u = 0; u < QUADS; ++u) read(v[u], first + u * 1024);
#pragma unroll
  for (int u = 0; u < QUADS; ++u) widen(mn, mx, v[u]);
  join(mn, mx, [] {});

  unsigned long long* const words = togetherWords + number % kTogetherTurns * (kTogetherWorkgroups * exchange::kWords);
  auto tell = [&](unsigned workgroup, float low, float high) __attribute__((always_inline)) {  // a thread a word, in one store
    const unsigned w = threadIdx.x;
    if (w < exchange::kWords)
      __hip_atomic_store(words + exchange::kWords * workgroup + w, exchange::word_of(number, __float_as_uint(w < 2 ? low : high), w % 2 != 0),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  tell(blockIdx.x, mn, mx);

  // Thread i hears workgroup i.
  const __amdgpu_buffer_rsrc_t source = __builtin_amdgcn_make_buffer_rsrc(words, 0, kTogetherWorkgroups * exchange::kWords * 8, 0x00020000);
  bool heard = threadIdx.x >= gridDim.x;
  auto ask = [&]() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");  // the words are asked for again each time
    unsigned long long theirs[exchange::kWords];
#pragma unroll
    for (unsigned w = 0; w < exchange::kWords; w += 2) {
      const together_v4u two = __builtin_amdgcn_raw_buffer_load_b128(source, 8 * (exchange::kWords * threadIdx.x + w), 0, kDeviceScope);
      theirs[w] = two[0] | (unsigned long long)two[1] << 32;
      theirs[w + 1] = two[2] | (unsigned long long)two[3] << 32;
    }
    heard = true;
#pragma unroll
    for (unsigned w = 0; w < exchange::kWords; ++w) heard = heard && exchange::belongs_to(theirs[w], number);
    if (heard) {
      mn = fminf(mn, __uint_as_float(exchange::value_of(theirs[0], theirs[1])));
      mx = fmaxf(mx, __uint_as_float(exchange::value_of(theirs[2], theirs[3])));
    }
  };
  if (!heard) {
    const unsigned long long start = wall_clock64();
    do ask();
    while (!heard && wall_clock64() - start < waitTicks);
  }
  while (true) {  // one part less is missing each time
    const unsigned long long silent = __ballot(!heard);
    join(mn, mx, [&] {
      if (threadIdx.x < kTogetherWorkgroups) shMissing[threadIdx.x >> 6] = silent;
    });
    unsigned missing = 0;
#pragma unroll
    for (unsigned w = 0; w < kTogetherWorkgroups / 64; ++w) missing += __popcll(shMissing[w]);
    if (missing == 0) break;  // the same for the whole workgroup
    unsigned part = 0, skip = blockIdx.x % missing;
    for (unsigned w = 0; w < kTogetherWorkgroups / 64; ++w) {
      unsigned long long left = shMissing[w];
      const unsigned here = __popcll(left);
      if (skip >= here) {
        skip -= here;
        continue;
      }
      while (skip-- > 0) left &= left - 1;
      part = 64 * w + __builtin_ctzll(left);
      break;
    }
    float low = kNoMinimum, high = kNoMaximum;
    for (int u = 0; u < QUADS; ++u) {
      float theirs[4];
      read(theirs, (size_t)part * (1024 * QUADS) + threadIdx.x + u * 1024);
      widen(low, high, theirs);
    }
    join(low, high, [] {});
    tell(part, low, high);
    if (threadIdx.x == part) {
      heard = true;
      mn = fminf(mn, low);
      mx = fmaxf(mx, high);
    }
    if (!heard) ask();
  }
  if (first == 0) {
    *mnOut = mn;
    *mxOut = mx;
  }
  const QuantizeScalars scalars = make_quantize_scalars(outType, mn, mx);
  const bool packed = scalars.r.bits == 8 && ((uintptr_t)out & 3u) == 0;
#pragma unroll
  for (int u = 0; u < QUADS; ++u) {
    const size_t i = first + u * 1024;
    if (i > total4 || (i == total4 && rest == 0)) break;
    long long q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) q[e] = quantize_one(v[u][e], scalars);
    if (packed && i < total4) {
      unsigned word = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) word |= ((unsigned)q[e] & 0xffu) << (8 * e);
      static_cast<unsigned*>(out)[i] = word;
    } else {
#pragma unroll
      for (unsigned e = 0; e < 4; ++e)
        if (i < total4 || e < rest) store_typed(out, outType, i * 4 + e, q[e]);
    }
  }
}

unsigned grid_for(size_t total, unsigned perThread = 1) {
  size_t blocks = (total + 256ull * perThread - 1) / (256ull * perThread);
  if (blocks > 256u * 32u) blocks = 256u * 32u;
  if (blocks < 1) blocks = 1;
  return (unsigned)blocks;
}

// The vector kernels: four 16-byte loads per thread per pass, at most 8 workgroups per CU; one load per thread while that
// still leaves CUs without work (131073 elements quantized: 32 workgroups against 129).
unsigned stream_grid(size_t total4) {
  size_t blocks = (total4 + 1023) / 1024;
  const size_t spread = (total4 + 255) / 256;
  if (blocks < 256) blocks = spread < 256 ? spread : 256;
  if (blocks > 256u * 8u) blocks = 256u * 8u;
  if (blocks < 1) blocks = 1;
  return (unsigned)blocks;
}

// The word on which a stream's range reductions count their workgroups; calls that get none reduce the partial results in a
// launch of its own.
StreamSlots gArrivalSlots(kArrivalSlots);

std::atomic<unsigned long long> gTogetherCalls{0};
constexpr int kDevices = 16;
quantize_exchange::LastStreams gTogetherStreams[kDevices];

// -1: unknown, or one of more than kDevices
int current_device() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return -1;
  }
  return dev < kDevices ? dev : -1;
}

// of a device, asked for once; 0: unknown
int compute_units(int dev) {
  static std::atomic<int> known[kDevices];
  if (dev < 0) return 0;
  int cus = known[dev].load(std::memory_order_relaxed);
  if (cus != 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  known[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

// Loads of a thread of the one launch; 0: the call takes the launches below.
unsigned together_quads(hipStream_t s, uint64_t total) {
  const int dev = current_device();
  const unsigned quads = quantize_exchange::quads_of(total, compute_units(dev));
  if (quads == 0 || !runs_in_order_now(s)) return 0;
  if (quads > 1 && gTogetherStreams[dev].with(s) > quantize_exchange::streams_of(quads)) return 0;
  return quads;
}

void launch_together(hipStream_t s, unsigned quads, const float* in, uint64_t total, void* out, int outType, float* mn, float* mx,
                     unsigned waitUs) {
  const unsigned long long number = quantize_exchange::number_of(gTogetherCalls.fetch_add(1, std::memory_order_relaxed));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)quantize_exchange::workgroups(total, quads)), dim3(1024), 0, s, in, (size_t)total, out, outType,
                       mn, mx, number, waitUs * 100ull);  // of the 100 MHz clock
  };
  if (quads == 1) launch(quantize_together_kernel<1>);
  else if (quads == 2) launch(quantize_together_kernel<2>);
  else if (quads == 4) launch(quantize_together_kernel<4>);
  else launch(quantize_together_kernel<8>);
}

bool valid_type(int t) { return t >= TFCC_ROCM_S8 && t <= TFCC_ROCM_U32; }

void launch_quantize(hipStream_t s, const float* in, uint64_t total, const float* minV, const float* maxV, void* out,
                     int outType, int fromData) {
  if ((outType == TFCC_ROCM_U8 || outType == TFCC_ROCM_S8) && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 4 == 0) {
    hipLaunchKernelGGL(quantize_8bit_vec_kernel, dim3(stream_grid(total / 4)), dim3(256), 0, s,
                       reinterpret_cast<const float4*>(in), (size_t)total, minV, maxV, static_cast<unsigned*>(out),
                       outType, fromData);
  } else {
    hipLaunchKernelGGL(quantize_kernel, dim3(grid_for(total)), dim3(256), 0, s, in, (size_t)total, minV, maxV, out,
                       outType, fromData);
  }
}

template <class T>
int reduce_rows(hipStream_t s, const void* a, unsigned batch, unsigned row, unsigned col, int* out) {
  unsigned long long rows = (unsigned long long)batch * row;
  if (rows >= (1ull << 31)) return set_error(TFCC_ROCM_INVALID_ARGUMENT, "reduce_sum: too many rows");
  unsigned blocks = (unsigned)((rows + 3) / 4);
  hipLaunchKernelGGL(reduce_rows_kernel<T>, dim3(blocks), dim3(256), 0, s, static_cast<const T*>(a),
                     (unsigned)rows, col, out);
  return check_launch("reduce_sum rows");
}

template <class T>
int reduce_cols(hipStream_t s, const void* a, unsigned batch, unsigned row, unsigned col, int* out) {
  size_t n = (size_t)batch * col;
  hipLaunchKernelGGL(zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, out, n);
  if (int e = check_launch("reduce_sum cols (zero)")) return e;
  if (batch > 65535) return set_error(TFCC_ROCM_INVALID_ARGUMENT, "reduce_sum: batch too large");
  if constexpr (sizeof(T) == 1) {
    if (col % 16 == 0 && (uintptr_t)a % 16 == 0 && row >= 64) {
      // slabs of at least 64 rows (sixteen 16-byte loads per thread), about a thousand workgroups where the
      // matrix is large enough
      const unsigned wideBlocks = (col / 16 + 63) / 64;
      unsigned wideSlabs = (1024 + wideBlocks * batch - 1) / (wideBlocks * batch);
      if (wideSlabs > row / 64) wideSlabs = row / 64;
      if (wideSlabs < 1) wideSlabs = 1;
      if (wideSlabs > 65535) wideSlabs = 65535;
      unsigned perSlab = (row + wideSlabs - 1) / wideSlabs;
      perSlab = (perSlab + 15) / 16 * 16;  // whole rounds of the four row lanes' four rows
      wideSlabs = (row + perSlab - 1) / perSlab;
      hipLaunchKernelGGL(reduce_cols_wide_kernel<T>, dim3(wideBlocks, wideSlabs, batch), dim3(256), 0, s,
                         static_cast<const T*>(a), row, col, perSlab, out);
      return check_launch("reduce_sum cols");
    }
  }
  const bool vec = sizeof(T) == 1 && col % 4 == 0 && (uintptr_t)a % 4 == 0;
  const unsigned colBlocks = vec ? (col / 4 + 255) / 256 : (col + 255) / 256;
  // enough row slabs for ~2048 workgroups
  unsigned slabs = (2048 + colBlocks * batch - 1) / (colBlocks * batch);
  if (slabs > (row + 31) / 32) slabs = (row + 31) / 32;
  if (slabs < 1) slabs = 1;
  if (slabs > 65535) slabs = 65535;
  const unsigned rowsPerSlab = (row + slabs - 1) / slabs;
  slabs = (row + rowsPerSlab - 1) / rowsPerSlab;
  if (vec)
    hipLaunchKernelGGL(reduce_cols_vec_kernel<T>, dim3(colBlocks, slabs, batch), dim3(256), 0, s,
                       static_cast<const T*>(a), row, col, rowsPerSlab, out);
  else
    hipLaunchKernelGGL(reduce_cols_kernel<T>, dim3(colBlocks, slabs, batch), dim3(256), 0, s,
                       static_cast<const T*>(a), row, col, rowsPerSlab, out);
  return check_launch("reduce_sum cols");
}

}  // namespace

int quantize_release_stream(hipStream_t stream) {
  int dev = 0;
  TFCC_HIP_CHECK(hipGetDevice(&dev));
  gArrivalSlots.release(dev, stream);
  return TFCC_ROCM_OK;
}

}  // namespace tfcc_rocm

using namespace tfcc_rocm;

extern "C" {

int tfcc_rocm_reduce_sum_rows(void* stream, const void* a, int type, unsigned batch, unsigned row,
                              unsigned col, int32_t* out) {
  TFCC_REQUIRE(a && out, "reduce_sum: null argument");
  TFCC_REQUIRE(batch > 0 && row > 0 && col > 0, "reduce_sum: empty tensor");
  switch (type) {
    case TFCC_ROCM_S8: return reduce_rows<int8_t>(as_stream(stream), a, batch, row, col, out);
    case TFCC_ROCM_U8: return reduce_rows<uint8_t>(as_stream(stream), a, batch, row, col, out);
    case TFCC_ROCM_S16: return reduce_rows<int16_t>(as_stream(stream), a, batch, row, col, out);
  }
  return set_error(TFCC_ROCM_INVALID_ARGUMENT, "reduce_sum: type %d (int8, uint8 or int16)", type);
}

int tfcc_rocm_reduce_sum_cols(void* stream, const void* a, int type, unsigned batch, unsigned row,
                              unsigned col, int32_t* out) {
  TFCC_REQUIRE(a && out, "reduce_sum: null argument");
  TFCC_REQUIRE(batch > 0 && row > 0 && col > 0, "reduce_sum: empty tensor");
  switch (type) {
    case TFCC_ROCM_S8: return reduce_cols<int8_t>(as_stream(stream), a, batch, row, col, out);
    case TFCC_ROCM_U8: return reduce_cols<uint8_t>(as_stream(stream), a, batch, row, col, out);
    case TFCC_ROCM_S16: return reduce_cols<int16_t>(as_stream(stream), a, batch, row, col, out);
  }
  return set_error(TFCC_ROCM_INVALID_ARGUMENT, "reduce_sum: type %d (int8, uint8 or int16)", type);
}

int tfcc_rocm_requantize(void* stream, const void* in, int in_type, void* out, int out_type,
                         uint64_t total, const float* min_in, const float* max_in,
                         const float* min_out, const float* max_out) {
  TFCC_REQUIRE(in && out && min_in && max_in && min_out && max_out, "requantize: null argument");
  TFCC_REQUIRE(total > 0, "requantize: empty tensor");
  TFCC_REQUIRE(valid_type(in_type) && valid_type(out_type), "requantize: bad type code");
  hipStream_t s = as_stream(stream);
  if (in_type == TFCC_ROCM_S32 && out_type == TFCC_ROCM_U8 && total % 4 == 0 && (uintptr_t)in % 16 == 0 &&
      (uintptr_t)out % 4 == 0) {
    hipLaunchKernelGGL(requantize_s32_u8_vec_kernel, dim3(stream_grid(total / 4)), dim3(256), 0, s,
                       static_cast<const int4*>(in), static_cast<unsigned*>(out), (size_t)(total / 4), min_in,
                       max_in, min_out, max_out);
  } else {
    hipLaunchKernelGGL(requantize_kernel, dim3(grid_for(total)), dim3(256), 0, s, in, in_type, out, out_type,
                       (size_t)total, min_in, max_in, min_out, max_out);
  }
  return check_launch("requantize");
}

int tfcc_rocm_dequantize(void* stream, const void* in, int in_type, uint64_t total,
                         const float* min_v, const float* max_v, float* out) {
  TFCC_REQUIRE(in && out && min_v && max_v, "dequantize: null argument");
  TFCC_REQUIRE(total > 0, "dequantize: empty tensor");
  TFCC_REQUIRE(valid_type(in_type), "dequantize: bad type code");
  if (in_type == TFCC_ROCM_S32 && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 16 == 0) {
    hipLaunchKernelGGL(dequantize_s32_vec_kernel, dim3(stream_grid(total / 4)), dim3(256), 0, as_stream(stream),
                       static_cast<const int4*>(in), (size_t)total, min_v, max_v, reinterpret_cast<float4*>(out));
  } else {
    hipLaunchKernelGGL(dequantize_kernel, dim3(grid_for(total)), dim3(256), 0, as_stream(stream), in, in_type,
                       (size_t)total, min_v, max_v, out);
  }
  return check_launch("dequantize");
}

int tfcc_rocm_quantize(void* stream, const float* in, uint64_t total, const float* min_v,
                       const float* max_v, void* out, int out_type) {
  TFCC_REQUIRE(in && out && min_v && max_v, "quantize: null argument");
  TFCC_REQUIRE(total > 0, "quantize: empty tensor");
  TFCC_REQUIRE(valid_type(out_type), "quantize: bad type code");
  launch_quantize(as_stream(stream), in, total, min_v, max_v, out, out_type, 0);
  return check_launch("quantize");
}

int tfcc_rocm_quantize_minmax(void* stream, const float* in, uint64_t total, void* out,
                              int out_type, float* min_v, float* max_v) {
  return tfcc_rocm_quantize_minmax_wait(stream, in, total, out, out_type, min_v, max_v, kTogetherWait);
}

int tfcc_rocm_quantize_minmax_wait(void* stream, const float* in, uint64_t total, void* out,
                                   int out_type, float* min_v, float* max_v, unsigned wait_us) {
  TFCC_REQUIRE(in && out && min_v && max_v, "quantize: null argument");
  TFCC_REQUIRE(total > 0, "quantize: empty tensor");
  TFCC_REQUIRE(valid_type(out_type), "quantize: bad type code");
  hipStream_t s = as_stream(stream);
  // In place (a four-byte type over its own input): only the form that writes nothing before the range is known, and then
  // every element where it was read.
  const uintptr_t inAt = (uintptr_t)in, outAt = (uintptr_t)out;
  const bool apart = inAt + 4 * total <= outAt || outAt + total * (int_range(out_type).bits / 8) <= inAt;
  const unsigned quads = apart && total > kWholeBest ? together_quads(s, total) : 0;
  if (quads != 0) {
    launch_together(s, quads, in, total, out, out_type, min_v, max_v, wait_us);
    return check_launch("quantize");
  }
  if (apart && total <= kWholeLimit) {
    hipLaunchKernelGGL(quantize_whole_kernel, dim3((unsigned)((total + 4095) / 4096)), dim3(1024), 0, s, in, (unsigned)total,
                       out, out_type, min_v, max_v);
    return check_launch("quantize");
  }
  unsigned* mnWord = reinterpret_cast<unsigned*>(min_v);
  unsigned* mxWord = reinterpret_cast<unsigned*>(max_v);
  if (apart && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 4 == 0) {
    // partial results, eight bytes per workgroup, rest in the output buffer until the quantize pass overwrites it
    float* partials = static_cast<float*>(out);
    int dev = 0;
    unsigned slot = 0;
    TFCC_HIP_CHECK(hipGetDevice(&dev));
    if (gArrivalSlots.of(dev, s, &slot)) {
      // one workgroup per CU at most: every arrival costs an atomic on one word and a write-back (192 workgroups of 256
      // threads for 786432 elements: 6 us, 48 of 1024: 5.6; so few come here on a GPU with few CUs only, the form above takes them on a whole one)
      const unsigned blocks = total >= 256u * 16384u ? 256u : (unsigned)((total + 16383) / 16384);
      hipLaunchKernelGGL((minmax_partial_kernel<16, true>), dim3(blocks), dim3(1024), 0, s, in, (size_t)total, partials, slot,
                         min_v, max_v);
    } else {
      const unsigned blocks = stream_grid(total / 4);
      hipLaunchKernelGGL((minmax_partial_kernel<4, false>), dim3(blocks), dim3(256), 0, s, in, (size_t)total, partials, 0u,
                         nullptr, nullptr);
      hipLaunchKernelGGL(minmax_final_kernel, dim3(1), dim3(256), 0, s, partials, blocks, min_v, max_v);
    }
  } else {
    hipLaunchKernelGGL(minmax_init_kernel, dim3(1), dim3(1), 0, s, mnWord, mxWord);
    hipLaunchKernelGGL(minmax_kernel, dim3(grid_for(total, 4)), dim3(256), 0, s, in, (size_t)total, mnWord, mxWord);
    hipLaunchKernelGGL(minmax_finish_kernel, dim3(1), dim3(1), 0, s, min_v, max_v);
  }
  launch_quantize(s, in, total, min_v, max_v, out, out_type, 1);
  return check_launch("quantize");
}

}  // extern "C"
