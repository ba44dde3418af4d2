// uint8 x int8 -> int32 products that are too small, too short or too ragged for the kernels with a pipeline of slabs:
// every byte is asked for at once and the wait for memory is paid about once.
//
// A product of 77 x 1001 x 1237 is 200 million operations and 1.3 MB: 0.1 us of matrix time and 0.3 us of traffic.  What
// it costs is latency, and a kernel that walks K slab by slab through LDS pays a trip to memory per slab (84 us in 128 x
// 128 tiles).  Here a workgroup owns BM x 64 outputs and its wavefronts deal the steps of 64 k among themselves; a
// wavefront has two steps in flight and nothing goes through LDS on the way in: the operand of A is 16 consecutive k of a
// row, loaded as it lies, and a lane turns its 16(k) x 4(n) bytes of B into operand order with byte permutes.  The
// partial tiles are added in LDS (integer adds: any order gives the same sum) and every thread finishes four columns.
//
// With a long K and few tiles one workgroup would make trip after trip to memory while most CUs have nothing to do (3 x
// 11304 x 910, fifteen tiles: 27 us): several workgroups share the tile's steps then, and add up in memory.
//
// Any K, N and alignment: buffer loads take any byte address, and those that would cross the end of an operand are moved
// back to end with it.  Arithmetic and epilogue
// are described in gemm_u8s8.hip (tfcc/mkl/operations/tfcc_mklquantization.cpp:33-69,176-201).
#include "common.hpp"
#include "gemv.hpp"
#include "qgemm_params.hpp"
#include "qgemm_small.hpp"
#include "qgemm_small_plan.hpp"
#include "stream_slots.hpp"

namespace tfcc_rocm {

typedef qgemm_v4i v4i;

namespace {

using qgemm_small_plan::kCols;
using qgemm_small_plan::kMaxResults;
using qgemm_small_plan::Plan;
using qgemm_small_plan::plan_of;
constexpr int kPitch = 68;   // words per tile row in LDS: the four row groups of a store fall on different banks

// The memory in which the workgroups that share a tile's K meet: a piece per stream, asked for by the first product that
// is split.  A word per result, the sum in its high half, how many have added to it in the low one; zero between launches.
int clear_words(hipStream_t stream, void* piece) { return tfcc_rocm_fill_async(stream, piece, 0, 8, kMaxResults); }
StreamPieces gPieces(kMaxResults * 8, 64, clear_words);  // 4 MB each

// The requantize scalars of the launch; the values themselves where the ranges lie in device memory.
__device__ __forceinline__ RequantScalars requant_scalars(const QGemmParams& p, float minC, float maxC) {
  if (p.minOut) return make_requant_scalars(TFCC_ROCM_S32, TFCC_ROCM_U8, minC, maxC, *p.minOut, *p.maxOut);
  RequantScalars rq;
  rq.inScale = p.inScale; rq.inMin = p.inMin; rq.outScale = p.outScale; rq.outOffset = p.outOffset;
  rq.inLowest = -2147483648LL; rq.outLowest = 0; rq.outHighest = 255; rq.mode = 0; rq.fillValue = 0;
  finish_requant_scalars(rq, 4294967295.0);
  return rq;
}
__device__ __forceinline__ void offsets_and_range(const QGemmParams& p, bool store, int& oA, int& oB, float& minC, float& maxC) {
  oA = p.offsetA;
  oB = p.offsetB;
  minC = maxC = 0.f;
  if (!p.minA) return;
  const float mnA = *p.minA, mxA = *p.maxA, mnB = *p.minB, mxB = *p.maxB;
  qmatmul_offsets(mnA, mxA, mnB, mxB, &oA, &oB);
  qmatmul_range(mnA, mxA, mnB, mxB, &minC, &maxC);
  if (store) {
    if (p.minC) *p.minC = minC;
    if (p.maxC) *p.maxC = maxC;
  }
}
__device__ __forceinline__ unsigned requantized(int v, const RequantScalars& rq) {
  const double off = (double)((unsigned)v ^ 0x80000000u);  // v - INT32_MIN
  if (rq.mode) return (unsigned)rq.fillValue;
  if (rq.fast32OK) return (unsigned)requantize_one_fast32(off, rq);
  if (rq.fastOK) return (unsigned)requantize_one_fast(off, rq);
  return (unsigned)requantize_one_exact((long long)v, rq);
}

// Operands shorter than one load of the kernels in slabs (16 bytes, so K below 16): a thread per result.
__global__ __launch_bounds__(256) void qgemm_tiny_kernel(const QGemmParams p, const QSmallOutputs o, unsigned long long total) {
  const unsigned long long i = (unsigned long long)blockIdx.x * 256 + threadIdx.x;
  int oA, oB;
  float minC, maxC;
  offsets_and_range(p, i == 0, oA, oB, minC, maxC);
  if (i >= total) return;
  const unsigned n = (unsigned)(i % p.N), m = (unsigned)(i / p.N % p.M), bi = (unsigned)(i / p.N / p.M);
  const unsigned char* A = p.A + (size_t)bi * p.strideA + (size_t)m * p.K;
  const signed char* B = p.B + (size_t)bi * p.strideB + n;
  unsigned sum = 0;
  for (unsigned k = 0; k < p.K; ++k) sum += (unsigned)((int)A[k] * (int)B[(size_t)k * p.N]);
  sum += (unsigned)oA * (unsigned)oB * p.K + (unsigned)p.rowsumA[(size_t)bi * p.strideRA + m] * (unsigned)oB +
         (unsigned)p.colsumB[(size_t)bi * p.strideRB + n] * (unsigned)oA;
  const size_t at = (size_t)bi * p.strideC + (size_t)m * p.N + n;
  if (p.C) p.C[at] = (int)sum;
  if (o.f32Out) o.f32Out[at] = (float)((double)(int)sum * ((double)o.scaleA * (double)o.scaleB[n]));
  if (p.Q) p.Q[at] = (unsigned char)requantized((int)sum, requant_scalars(p, minC, maxC));
}

template <int BM, int WAVES, bool SHARED>
__global__ __launch_bounds__(WAVES * 64) void qgemm_small_kernel(const QGemmParams p, const QSmallOutputs o, unsigned splits,
                                                                 unsigned long long* meeting) {
  constexpr int kThreads = WAVES * 64, RB = BM / 16, WORKERS = WAVES - 1;
  __shared__ int tile[BM * kPitch];
  __shared__ int sums[kCols];
  __shared__ struct {
    RequantScalars rq;
    int offsetA, offsetB;
    unsigned row[BM];  // sums of the tile's rows of A
    alignas(16) unsigned col[kCols];  // and columns of B as the caller gave them
    alignas(16) float scale[kCols];
  } shared;
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  for (int i = tid; i < BM * kPitch; i += kThreads) tile[i] = 0;
  if (tid < kCols) sums[tid] = 0;

  unsigned tm, tn, bi, tileIndex;
  {
    // each XCD a contiguous run of tiles, the tiles of one column block next to each other: B is the larger operand
    const unsigned xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    const unsigned L = xcd * p.chunk + slot;
    if (slot >= p.chunk || L >= p.tilesTotal) return;
    tileIndex = L;
    bi = udiv_apply(L, p.perBatchMagic, p.perBatchShift);
    const unsigned t = L - bi * (p.tilesM * p.tilesN);
    tn = udiv_apply(t, p.bandMagic, p.bandShift);  // here: division by tilesM
    tm = t - tn * p.tilesM;
  }
  const unsigned m0 = tm * BM, n0 = tn * kCols;
  const unsigned M = p.M, N = p.N, K = p.K;
  const unsigned sizeA = M * K, sizeB = K * N;
  const __amdgpu_buffer_rsrc_t rsrcA = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<unsigned char*>(p.A + (size_t)bi * p.strideA), 0, (int)sizeA, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrcB = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<signed char*>(p.B + (size_t)bi * p.strideB), 0, (int)sizeB, 0x00020000);
  __syncthreads();  // the tile is clear; passed before the loads are asked for, whose return it would wait for

  // What the finish needs besides the sums.  The requantize scalars are a few hundred double operations: the last
  // wavefront works them out for all while the operands travel, and does nothing else (next to loads in flight they
  // would cost every wavefront the registers for both).  It also fetches the caller's sums and scales: behind the operands they
  // would be a trip to memory of their own (200 x 500 x 300 5.15 -> 4.97 us), and in front of them they hold them up.
  auto prepare = [&]() __attribute__((always_inline)) {
    static_assert(BM <= 64 && kCols == 64, "a lane has one of each");
    unsigned row = 0, col = 0;
    float scale = 0.f;
    if (!SHARED && lane < BM && m0 + lane < M) row = (unsigned)p.rowsumA[(size_t)bi * p.strideRA + m0 + lane];
    if (!SHARED && n0 + lane < N) {
      col = (unsigned)p.colsumB[(size_t)bi * p.strideRB + n0 + lane];
      if (o.f32Out) scale = o.scaleB[n0 + lane];
    }
    int oA, oB;
    float minC, maxC;
    offsets_and_range(p, blockIdx.x == 0 && (!SHARED || blockIdx.y == 0) && lane == 0, oA, oB, minC, maxC);
    if (lane == 0) {
      shared.offsetA = oA;
      shared.offsetB = oB;
    }
    if (p.Q) {
      const RequantScalars rq = requant_scalars(p, minC, maxC);
      if (lane == 0) shared.rq = rq;
    }
    if constexpr (!SHARED) {
      if (lane < BM) shared.row[lane] = row;
      shared.col[lane] = col;
      shared.scale[lane] = scale;
    }
  };

  // (Where several workgroups share a tile, every thread has its own four results' in registers, in front of the operands:
  // 11 x 5248 x 512 5.8 -> 5.3 us, through LDS 5.75; elsewhere that way is the slower one, 15 x 163 x 264 4.05 -> 4.3.)
  unsigned ownRow = 0, ownCol[4] = {};
  float ownScale[4] = {};
  if constexpr (SHARED) {
    static_assert(!SHARED || BM * 16 <= kThreads, "a thread finishes four results");
    const unsigned grow = m0 + (tid >> 4), gcol = n0 + 4 * (tid & 15);
    const bool in = tid < BM * 16 && grow < M;
    if (in) ownRow = (unsigned)p.rowsumA[(size_t)bi * p.strideRA + grow];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (in && gcol + e < N) ownCol[e] = (unsigned)p.colsumB[(size_t)bi * p.strideRB + gcol + e];
      if (in && gcol + e < N && o.f32Out) ownScale[e] = o.scaleB[gcol + e];
    }
  }

  // the workers of all workgroups that share the tile deal its steps among themselves
  const unsigned steps = (K + 63) / 64, workers = SHARED ? splits * WORKERS : WORKERS, first = (SHARED ? blockIdx.y * WORKERS : 0u) + wave;
  const unsigned offA = (m0 + j) * K + kg * 16, offB = kg * 16 * N + n0 + j * 4;
  v4i acc[RB][4];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[i][e] = v4i{0, 0, 0, 0};
  int colsum[4] = {0, 0, 0, 0};

  // Every load is moved back far enough to end inside its operand.  That changes the bytes only of what crosses the end
  // or lies behind it, and those are put right.  For A that is the step in which K ends (and the one behind it that evens
  // out a pair).  A load of B crosses the end from the last three rows on if N is 1, from the last row on otherwise, so
  // the step that holds row K - 3 counts too: with K = 64 i + 1 or 64 i + 2 it is the step before.  (Rows of A past M and
  // columns of B past N hold whatever they hold: they are not stored.)
  const unsigned lastA = sizeA - 16, lastB = sizeB - 4;
  if (wave == WORKERS) prepare();
  else for (unsigned s = first; s < steps; s += 2 * workers) {
    v4i a[2][RB];
    unsigned b[2][16];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const unsigned ka = offA + (s + u * workers) * 64, kb = offB + (s + u * workers) * 64 * N;
#pragma unroll
      for (int q = 0; q < 16; ++q) b[u][q] = __builtin_amdgcn_raw_buffer_load_b32(rsrcB, min(kb + q * N, lastB), 0, 0);
#pragma unroll
      for (int i = 0; i < RB; ++i)
        a[u][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrcA, min(ka + i * 16 * K, lastA), 0, 0));
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const unsigned step = s + u * workers;
      if ((step + 1) * 64 + 3 > K) {
        unsigned ka = offA + step * 64, kb = offB + step * 64 * N;
        asm volatile("" : "+v"(ka), "+v"(kb));  // worked out again, instead of keeping every load's offset in a register
#pragma unroll
        for (int q = 0; q < 16; ++q) b[u][q] = moved4(b[u][q], max(kb + q * N, lastB) - lastB);
#pragma unroll
        for (int i = 0; i < RB; ++i) a[u][i] = moved16(a[u][i], max(ka + i * 16 * K, lastA) - lastA);
      }
      unsigned col[4][4];  // [column][k quad]
#pragma unroll
      for (int kq = 0; kq < 4; ++kq) {
        unsigned c4[4];
        transpose4x4(&b[u][4 * kq], c4);
#pragma unroll
        for (int e = 0; e < 4; ++e) col[e][kq] = c4[e];
      }
#pragma unroll
      for (int i = 0; i < RB; ++i) a[u][i] = a[u][i] ^ (int)0x80808080;  // a' = a - 128
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const v4i bv = {(int)col[e][0], (int)col[e][1], (int)col[e][2], (int)col[e][3]};
#pragma unroll
        for (int i = 0; i < RB; ++i) acc[i][e] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[u][i], bv, acc[i][e], 0, 0, 0);
        if (!p.colsumExact) {
#pragma unroll
          for (int kq = 0; kq < 4; ++kq) colsum[e] = __builtin_amdgcn_sdot4((int)col[e][kq], 0x01010101, colsum[e], false);
        }
      }
    }
  }

  // lane (j, kg) holds rows 16 i + 4 kg + r of column 4 j + e; column 4 j + e lies at word e * 16 + j of its tile row
  if (wave < WORKERS && first < steps) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) atomicAdd(&tile[(16 * i + 4 * kg + r) * kPitch + e * 16 + j], acc[i][e][r]);
    if (!p.colsumExact) {
#pragma unroll
      for (int e = 0; e < 4; ++e) atomicAdd(&sums[e * 16 + j], colsum[e]);
    }
  }
  __syncthreads();

  const unsigned offsetA = (unsigned)shared.offsetA, offsetB = (unsigned)shared.offsetB, global = offsetA * offsetB * K;
  for (int idx = tid; idx < BM * 16; idx += kThreads) {
    const int row = idx >> 4, c = idx & 15;
    const unsigned grow = m0 + row, gcol = n0 + 4 * c;
    if (grow >= M || gcol >= N) continue;
    const unsigned rt = global + (SHARED ? ownRow : shared.row[row]) * offsetB;
    const size_t at = (size_t)bi * p.strideC + (size_t)grow * N + gcol;
    const unsigned left = N - gcol;
    unsigned cs[4], sum[4];
    bool mine[4];  // the results that this thread finishes
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      mine[e] = e < (int)left;
      cs[e] = SHARED ? ownCol[e] : shared.col[4 * c + e];
      sum[e] = (unsigned)tile[row * kPitch + e * 16 + c] + (p.colsumExact ? 0u : 128u * (unsigned)sums[e * 16 + c]);
    }
    if constexpr (SHARED) {
      // One trip to memory and back, no fences: what an addition returns says whether it was the last one, and then it
      // holds the sum of the others (whole numbers: in any order the same).
      unsigned long long* const words = meeting + (size_t)tileIndex * (BM * kCols) + idx;
      unsigned long long before[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (mine[e])
          before[e] = __hip_atomic_fetch_add(words + e * (BM * 16), ((unsigned long long)sum[e] << 32) | 1ull, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        mine[e] = mine[e] && (unsigned)before[e] == splits - 1;
        if (!mine[e]) continue;
        sum[e] += (unsigned)(before[e] >> 32);
        __hip_atomic_store(words + e * (BM * 16), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if (!(mine[0] | mine[1] | mine[2] | mine[3])) continue;
    }
    int v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (int)(sum[e] + (p.colsumExact ? 128u * cs[e] : 0u) + cs[e] * offsetA + rt);
    const bool four = (mine[0] & mine[1] & mine[2] & mine[3]) && p.vectorStores;
    if (p.C) {
      if (four) *reinterpret_cast<v4i*>(p.C + at) = v4i{v[0], v[1], v[2], v[3]};
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (mine[e]) p.C[at + e] = v[e];
    }
    if (o.f32Out) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (mine[e]) o.f32Out[at + e] = (float)((double)v[e] * ((double)o.scaleA * (double)(SHARED ? ownScale[e] : shared.scale[4 * c + e])));
    }
    if (p.Q) {
      const RequantScalars& rq = shared.rq;
      unsigned q[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) q[e] = requantized(v[e], rq);
      if (four) *reinterpret_cast<unsigned*>(p.Q + at) = q[0] | (q[1] << 8) | (q[2] << 16) | (q[3] << 24);
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (mine[e]) p.Q[at + e] = (unsigned char)q[e];
    }
  }
}

template <int BM, int WAVES, bool SHARED = false>
int launch(hipStream_t stream, QGemmParams p, const QSmallOutputs& o, unsigned splits = 1, unsigned long long* meeting = nullptr) {
  p.tilesM = (p.M + BM - 1) / BM;
  p.tilesN = (p.N + kCols - 1) / kCols;
  const unsigned long long total = (unsigned long long)p.tilesM * p.tilesN * p.batch;
  if (total > 0x7fffffffull) return set_error(TFCC_ROCM_INVALID_ARGUMENT, "quantized matmul: too many tiles");
  p.tilesTotal = (unsigned)total;
  p.chunk = (p.tilesTotal + 7) / 8;
  const UDiv perBatch = udiv_prepare(p.tilesM * p.tilesN), rows = udiv_prepare(p.tilesM);
  p.perBatchMagic = perBatch.magic; p.perBatchShift = perBatch.shift;
  p.bandMagic = rows.magic; p.bandShift = rows.shift;
  hipLaunchKernelGGL((qgemm_small_kernel<BM, WAVES, SHARED>), dim3(p.chunk * 8, splits), dim3(WAVES * 64), 0, stream, p, o, splits, meeting);
  return check_launch("quantized matmul (small)");
}

unsigned long long* meeting_of(hipStream_t stream) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  return static_cast<unsigned long long*>(gPieces.of(dev, stream));
}

}  // namespace

void qgemm_small_release_stream(int dev, hipStream_t stream) { gPieces.release(dev, stream); }

bool qgemm_small_supported(const QGemmParams& p) {
  return ((unsigned long long)p.M + 64) * p.K + 4096 < (1ull << 31) && ((unsigned long long)p.K + 4160) * p.N + 4096 < (1ull << 31);
}

bool qgemm_small_splits(hipStream_t stream, unsigned m, unsigned n, unsigned k, unsigned instead) {
  const Plan plan = plan_of(m, n, k, 1);
  return plan.splits > 1 && plan.splitCost + 70 <= instead && meeting_of(stream) != nullptr;
}

int qgemm_small_launch(hipStream_t stream, QGemmParams p, const QSmallOutputs& o, bool split) {
  if ((unsigned long long)p.M * p.K < 16 || (unsigned long long)p.K * p.N < 16) {
    const unsigned long long total = (unsigned long long)p.M * p.N * p.batch;
    if ((total + 255) / 256 > 0x7fffffffull) return set_error(TFCC_ROCM_INVALID_ARGUMENT, "quantized matmul: too many results");
    hipLaunchKernelGGL(qgemm_tiny_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, p, o, total);
    return check_launch("quantized matmul (tiny)");
  }
  p.vectorStores = p.N % 4 == 0 && p.strideC % 4 == 0 && (uintptr_t)p.C % 16 == 0 && (uintptr_t)p.Q % 4 == 0;
  const Plan plan = plan_of(p.M, p.N, p.K, p.batch);
  if (unsigned long long* const meeting = plan.splits > 1 && (split || plan.better) ? meeting_of(stream) : nullptr)
    return plan.splitWaves == 4 ? launch<16, 4, true>(stream, p, o, plan.splits, meeting) : launch<16, 8, true>(stream, p, o, plan.splits, meeting);
  if (plan.rows == 64) return plan.waves == 4 ? launch<64, 4>(stream, p, o) : launch<64, 8>(stream, p, o);
  if (plan.rows == 32) return plan.waves == 4 ? launch<32, 4>(stream, p, o) : launch<32, 8>(stream, p, o);
  return plan.waves == 4 ? launch<16, 4>(stream, p, o) : plan.waves == 8 ? launch<16, 8>(stream, p, o) : launch<16, 16>(stream, p, o);
}

}  // namespace tfcc_rocm
