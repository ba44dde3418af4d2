// fp32 products of some hundred results a CU and a long K: few tiles for the kernels that walk K in slabs, whose four K groups then
// multiply for 10 us and more on a part of the CUs (128 x 3072 x 768 has 96 tiles of 32 x 32), and many small ones for the kernel of
// 16 x 16 tiles, which asks for every operand twice as often as 32 x 32 do.
//
// A workgroup owns 32 rows and one or two blocks of 32 columns and deals the steps of K (16 k each) among eight wavefronts, and
// several workgroups share a tile's steps where that fills the chip.  Nothing is shared before the partial tiles meet, so nothing goes
// through LDS on the way in: a lane loads its operands of the 32x32x2 matrix op as they lie, eight consecutive k of a row of A in
// two loads, and of each of eight rows of B one word, or two neighbouring ones (the blocks' columns alternate).  Four
// or two steps are on their way at once; more make the first one wait longer (128 x 3072 x 768 13.1 -> 13.4 us), since the launch is bound
// by what the L2s hand out: 32 x 64 tiles of 614 k are 240 KB for each CU, 5 us, where the matrix ops take 4.3.  Tiles of 32 x 128
// were no better (fewer workgroups, or more splits to meet).
//
// us, before (the kernels of sgemm_wave96.hip and sgemm_skinny.hip) -> now: 128 x 3072 x 768 19.1 -> 13.1, 128 x 4096 x 1024 24.6 -> 16.2, 64 x 2373 x
// 1536 17.6 -> 11.3, 256 x 2048 x 512 13.5 -> 10.3, 96 x 7608 x 824 30.8 -> 19.5, 75 x 4928 x 1344 29.3 -> 18.4.
//
// An element is the sum of its wavefronts' partial sums, added in the order of the wavefronts, then of the splits; wavefront w of
// W has the steps w, w + W, ..., dealt in ascending order to four accumulators.  Against float64 that leaves a quarter of the
// error of four K groups (75 x 4928 x 1344 5.2e-7 -> 1.2e-7) and 0.8 to 1.0 of that of the 16 x 16 tiles.  B transposed and B as stored give the
// same bits, and so does a launch that may not use the memory in which the splits meet (a stream that is being captured): its
// workgroups take all splits of a tile, one after the other.  Bias, residual and the erf-form GELU follow as in the other kernels
// (tfcc/mkl/interfaces/tfcc_mklblasinterface.cpp:41-67, 69-78, 87-118).
#include <type_traits>

#include "common.hpp"
#include "sgemm_deal_plan.hpp"
#include "sgemm_params.hpp"
#include "stream_slots.hpp"

namespace tfcc_rocm {
namespace {

using sgemm_detail::SgemmParams;
using sgemm_deal_plan::kMaxParts;
using sgemm_deal_plan::kStep;
using sgemm_deal_plan::kWaves;

typedef float deal_v16f __attribute__((ext_vector_type(16)));

// The memory in which the splits of a tile meet, a piece per stream.
constexpr unsigned kMaxGroups = 3, kMaxTiles = kMaxGroups * kMaxParts / 2048;  // tiles of products that are split, at least in two
struct Meeting {
  float partials[(size_t)kMaxGroups * kMaxParts];
  unsigned counts[kMaxTiles];  // zero between launches: the workgroup that arrives last sees to it
};
int clear_counts(hipStream_t stream, void* piece) {
  return tfcc_rocm_fill_async(stream, static_cast<Meeting*>(piece)->counts, 0, sizeof(unsigned), kMaxTiles);
}
StreamPieces gPieces(sizeof(Meeting), 64, clear_counts);  // 12 MB each

// ALONE: the workgroup has all splits of its tile, in two teams of eight wavefronts that take turns; the partial tiles of four splits
// wait in LDS.  Replayed from a graph, the kernels of sgemm_wave96.hip and sgemm_skinny.hip -> this one: 75 x 4928 x 1344 29.5 -> 30.2
// us, 96 x 7608 x 824 47.7 -> 46.6, 24 x 3183 x 2827 21.2 -> 23.9, 128 x 2384 x 992 16.7 -> 14.2, 466 x 5928 x 288 36.5 -> 32.9, 128 x 3072 x 768
// 19.4 -> 23.5, 75 x 3072 x 832 19.4 -> 18.4, 369 x 1220 x 170 10.0 -> 11.5 (one team: 47, 69, 36, 16, 50, 38, 21 and 13).  Bound by what one CU
// loads: the last of an odd number of splits shared by both teams took 1.02 to 1.1 of the time, one team with eight steps on their way
// across the splits' borders 1.06 to 1.3 (256 x 2048 x 512 13.4 -> 16.4).  Which products that loses too much for: sgemm_deal_plan.hpp.
template <int NB, bool TRANSB, bool ALONE, class Arguments>
__global__ __launch_bounds__(64 * kWaves * (ALONE ? 2 : 1), ALONE ? 4 : 2) void sgemm_deal_kernel(const float* hotA, const float* hotB, unsigned M, unsigned N, unsigned K,
                                                                    unsigned lda, unsigned ldb, unsigned tilesM, unsigned tilesTotal,
                                                                    unsigned chunk, unsigned splits, unsigned perWave, Meeting* meeting,
                                                                    const Arguments arguments) {
  const SgemmParams p = arguments.whole();
  static_assert(NB == 1 || NB == 2, "a lane's columns of a row of B in one load");
  constexpr bool GROUPED = std::is_same<Arguments, SgemmParams>::value;
  constexpr int TEAMS = ALONE ? 2 : 1, THREADS = 64 * kWaves * TEAMS;
  constexpr int SETS = NB == 1 && !ALONE ? 4 : 2, ACCS = 4, ROWS = 1024 / THREADS, OUT = NB * ROWS;  // steps on their way, results that a thread finishes
  constexpr unsigned HELD = ALONE ? 4 : 1;  // splits that wait in LDS
  __shared__ float part[HELD][kWaves][NB * 16 * 64];
  __shared__ unsigned arrived;
  const unsigned tid = threadIdx.x, lane = tid & 63;
  const unsigned waveInGroup = __builtin_amdgcn_readfirstlane(tid >> 6), team = waveInGroup / kWaves, wave = waveInGroup % kWaves;
  // each XCD gets a contiguous run of tiles, the row tiles of a column tile side by side: they read the same piece of B
  const unsigned L = (blockIdx.x & 7u) * chunk + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= chunk || L >= tilesTotal) return;
  const unsigned tn = L / tilesM, tm = L - tn * tilesM, group = blockIdx.y;
  const unsigned m0 = tm * 32, n0 = tn * 32 * NB;
  const float* A = hotA;
  const float* B = GROUPED && p.groups ? p.groupB[group] : hotB;

  // A lane has row lane % 32, NB consecutive columns from NB (lane % 32) on, and eight consecutive k of a step's sixteen.  Rows past
  // the edge read the last one, and their sums are dropped; words past the end of an operand read zeros.
  const unsigned g = lane >> 5, edge = lane & 31u;
  const unsigned row = min(m0 + edge, M - 1), aOff = (row * lda + 8 * g) * 4u;
  unsigned bOff[TRANSB ? NB : 8];
  if (TRANSB) {
#pragma unroll
    for (int j = 0; j < NB; ++j) bOff[j] = (min(n0 + NB * edge + j, N - 1) * ldb + 8 * g) * 4u;
  } else {
#pragma unroll
    for (unsigned s = 0; s < 8; ++s) bOff[s] = ((8 * g + s) * ldb + min(n0 + NB * edge, N - 1)) * 4u;
  }
  const unsigned bytesA = ((M - 1) * lda + K) * 4u, bytesB = TRANSB ? ((N - 1) * ldb + K) * 4u : ((K - 1) * ldb + N) * 4u;
  struct Ops { float a[8], b[NB][8]; };
  auto load = [&](Ops& o, unsigned step) __attribute__((always_inline)) {
    // the step's k goes into the descriptors, base up and size down, so that the range check sees all of an offset
    const unsigned k = step * kStep, skipB = (TRANSB ? k : k * ldb) * 4u;
    const __amdgpu_buffer_rsrc_t rsrcA = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A) + k, 0, (int)(bytesA - k * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcB = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(B)) + skipB, 0, (int)(bytesB - skipB), 0x00020000);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const auto a = __builtin_amdgcn_raw_buffer_load_b128(rsrcA, aOff + 16 * h, 0, 0);
      __builtin_memcpy(o.a + 4 * h, &a, 16);
    }
    if constexpr (TRANSB) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const auto b = __builtin_amdgcn_raw_buffer_load_b128(rsrcB, bOff[j] + 16 * h, 0, 0);
          __builtin_memcpy(o.b[j] + 4 * h, &b, 16);
        }
    } else {
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        float b[NB];
        if constexpr (NB == 1) {
          const auto w = __builtin_amdgcn_raw_buffer_load_b32(rsrcB, bOff[s], 0, 0);
          __builtin_memcpy(b, &w, 4);
        } else {
          const auto w = __builtin_amdgcn_raw_buffer_load_b64(rsrcB, bOff[s], 0, 0);
          __builtin_memcpy(b, &w, 8);
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) o.b[j][s] = b[j];
      }
    }
  };
  // of the step in which K ends: past it a row of A, and of B transposed, goes on with the next one
  auto mask = [&](Ops& o, unsigned step) __attribute__((always_inline)) {
#pragma unroll
    for (unsigned s = 0; s < 8; ++s) {
      const bool in = step * kStep + 8 * g + s < K;
      o.a[s] = in ? o.a[s] : 0.f;
      if (TRANSB) {
#pragma unroll
        for (int j = 0; j < NB; ++j) o.b[j][s] = in ? o.b[j][s] : 0.f;
      }
    }
  };
  const unsigned total = (K + kStep - 1) / kStep, lanes = splits * kWaves;  // wavefronts that share the tile
  const unsigned oneMore = total - perWave * lanes;

  // what the finish needs: thread t finishes words t, t + THREADS, ... of each block as the accumulators hold it
  float bv[NB], rv[OUT];
  // value q: word t + THREADS (q / NB) of block q % NB
  auto rowOf = [&](int q) __attribute__((always_inline)) { const unsigned r = (tid + THREADS * (q / NB)) >> 6; return m0 + 8 * (r >> 2) + 4 * g + (r & 3u); };
  auto colOf = [&](int q) __attribute__((always_inline)) { return n0 + NB * edge + q % NB; };
  auto mine = [&](int q) __attribute__((always_inline)) { return rowOf(q) < M && colOf(q) < N; };
  auto loadFinish = [&]() __attribute__((always_inline)) {
    const float* bias = GROUPED && p.groups ? p.groupBias[group] : p.bias;
#pragma unroll
    for (int q = 0; q < OUT; ++q) {
      if (q < NB) bv[q] = bias && colOf(q) < N ? bias[colOf(q)] : 0.f;
      rv[q] = p.residual && mine(q) ? p.residual[(size_t)rowOf(q) * N + colOf(q)] : 0.f;
    }
  };

  float v[OUT];
  // Step i of a wavefront is in set i % SETS.  What is under way is the same on every path, or the compiler would wait for
  // every load before it uses the first: behind the last step that step is asked for again.
  Ops ops[SETS];
  auto loadFirst = [&](unsigned split) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < SETS; ++u) load(ops[u], min(split * kWaves + wave + u * lanes, total - 1));
  };
  auto sumSplit = [&](unsigned split, unsigned held) __attribute__((always_inline)) {
    const unsigned first = split * kWaves + wave;
    const unsigned steps = perWave + (first < oneMore ? 1u : 0u);
    deal_v16f acc[ACCS][NB];
#pragma unroll
    for (int u = 0; u < ACCS; ++u)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][j][r] = 0.f;
    auto multiply = [&](const Ops& o, int u) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[u][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(o.a[s], o.b[j][s], acc[u][j], 0, 0, 0);
    };
    auto loadStep = [&](int set, unsigned i) __attribute__((always_inline)) {
      load(ops[set], min(first + i * lanes, total - 1));
    };
    // the last step of the wavefront that has it is masked, outside the loop
    const bool ends = K % kStep != 0 && (total - 1) % lanes == first;
    unsigned i = 0;
    for (; i + ACCS < steps; i += ACCS) {
#pragma unroll
      for (int u = 0; u < ACCS; ++u) {
        multiply(ops[u % SETS], u);
        loadStep(u % SETS, i + SETS + u);
        __builtin_amdgcn_sched_barrier(0);  // or the compiler waits for all sets before it asks for any again
      }
    }
#pragma unroll
    for (int u = 0; u < ACCS; ++u)
      if (i + u < steps) {
        if (ends && i + u + 1 == steps) mask(ops[u % SETS], total - 1);
        multiply(ops[u % SETS], u);
        if (u + SETS < ACCS) loadStep(u % SETS, i + SETS + u);
      }
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[held][wave][(j * 16 + r) * 64 + lane] = (acc[0][j][r] + acc[1][j][r]) + (acc[2][j][r] + acc[3][j][r]);
  };
  auto meet = [&](unsigned held, bool first) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < OUT; ++q) {
      const unsigned at = q % NB * 1024 + q / NB * THREADS + tid;
      float sum = part[held][0][at];
#pragma unroll
      for (unsigned w = 1; w < kWaves; ++w) sum += part[held][w][at];
      v[q] = first ? sum : v[q] + sum;
    }
  };
  if constexpr (ALONE) {
    loadFinish();
    for (unsigned held = 0; held < splits; held += HELD) {
      if (held) __syncthreads();
#pragma unroll 1
      for (unsigned split = team; split < HELD && held + split < splits; split += TEAMS) {
        loadFirst(held + split);
        sumSplit(held + split, split);
      }
      __syncthreads();
      for (unsigned split = 0; split < HELD && held + split < splits; ++split) meet(split, held + split == 0);
    }
  } else {
    loadFirst(blockIdx.z);
    loadFinish();
    sumSplit(blockIdx.z, 0);
    __syncthreads();
    meet(0, true);
    if (splits > 1) {
      // The partial tile goes past the caches, and waiting for the stores is all the order there has to be in front of the
      // count; the workgroup that arrives last adds the partial tiles in the order of the splits.
      constexpr unsigned TILE = NB * 1024;
      const unsigned tile = group * tilesTotal + L;
      float* const at = meeting->partials + (size_t)tile * splits * TILE + tid;
      unsigned* const count = meeting->counts + tile;
#pragma unroll
      for (int q = 0; q < OUT; ++q)
        __hip_atomic_store(at + blockIdx.z * TILE + THREADS * q, v[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) arrived = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      if (arrived != splits - 1) return;
      if (tid == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int q = 0; q < OUT; ++q) v[q] = __hip_atomic_load(at + THREADS * q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (unsigned s = 1; s < splits; ++s) {
#pragma unroll
        for (int q = 0; q < OUT; ++q) v[q] += __hip_atomic_load(at + s * TILE + THREADS * q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  float* C = GROUPED && p.groups ? p.groupC[group] : p.C;
#pragma unroll
  for (int q = 0; q < OUT; ++q) {
    if (!mine(q)) continue;
    float x = v[q] + bv[q % NB];
    if (p.residual) x += rv[q];
    if (p.act == 1) x = gelu_erf_f32(x);
    C[(size_t)rowOf(q) * p.ldc + colOf(q)] = x;
  }
}

template <int NB, bool TRANSB>
int launch_deal(hipStream_t stream, SgemmParams p, unsigned splits) {
  const unsigned groups = p.groups ? p.groups : 1u;
  p.batch = 1;
  if (!sgemm_detail::set_tiles(p, 32, 32 * NB)) return set_error(TFCC_ROCM_INVALID_ARGUMENT, "sgemm: too many tiles");
  Meeting* meeting = nullptr;
  if (splits > 1 && (unsigned long long)groups * p.tilesTotal * splits * NB * 1024 <= (unsigned long long)kMaxGroups * kMaxParts) {
    int dev = 0;
    TFCC_HIP_CHECK(hipGetDevice(&dev));
    meeting = static_cast<Meeting*>(gPieces.of(dev, stream));
  }
  const bool alone = splits > 1 && meeting == nullptr;  // then in tiles of one block: their number, not that of the splits, fills the chip
  if (alone && !sgemm_detail::set_tiles(p, 32, 32)) return set_error(TFCC_ROCM_INVALID_ARGUMENT, "sgemm: too many tiles");
  auto launch = [&](const auto& arguments) {
    using Arguments = std::decay_t<decltype(arguments)>;
    auto kern = alone ? sgemm_deal_kernel<1, TRANSB, true, Arguments> : sgemm_deal_kernel<NB, TRANSB, false, Arguments>;
    hipLaunchKernelGGL(kern, dim3(p.chunk * 8, groups, alone ? 1u : splits), dim3(64 * kWaves * (alone ? 2 : 1)), 0, stream, p.A, p.B, p.M,
                       p.N, p.K, p.lda, p.ldb, p.tilesM, p.tilesTotal, p.chunk, splits, (p.K + kStep - 1) / kStep / (splits * kWaves),
                       meeting, arguments);
  };
  if (p.groups) launch(p);
  else launch(sgemm_detail::SgemmFinish(p));
  return check_launch("sgemm");
}

}  // namespace

namespace sgemm_detail {

int sgemm_deal_launch(hipStream_t stream, const SgemmParams& p, unsigned splits, unsigned blocks, bool transB) {
  if (transB) return blocks == 1 ? launch_deal<1, true>(stream, p, splits) : launch_deal<2, true>(stream, p, splits);
  return blocks == 1 ? launch_deal<1, false>(stream, p, splits) : launch_deal<2, false>(stream, p, splits);
}

void sgemm_deal_release_stream(int dev, hipStream_t stream) { gPieces.release(dev, stream); }

}  // namespace sgemm_detail
}  // namespace tfcc_rocm
