// fp32 products whose tiles leave most of the chip idle: few rows, K long against N.  In 32-row tiles 32 x 3072 x 768 is
// 24 workgroups of four wavefronts, each walking a quarter of K slab by slab; the matrix cores of 24 CUs and their loads
// decide (19 us for 9 MB of B).
//
// A workgroup owns 16 (or 32) rows x 16 columns and deals the steps of K (16 k each) among eight wavefronts; where the tiles leave
// CUs without work, several workgroups share a tile's steps.  Nothing is shared before the partial tiles meet, so nothing
// goes through LDS on the way in: a lane loads its operands of the 16x16x4 matrix op as they lie, four consecutive k of a
// row of A in one load and the same four k of its column of B, with two batches of four steps under way.  Bound by what a
// CU can have on its way from memory.  (Tiles of 16 x 32, whole lines of B, take twice as long: half the workgroups.)
//
// With weights from memory, against the tiles of 32 rows: 32 x 3072 x 768 19.6 -> 8.6 us,
// 9 x 4096 x 1024 24.3 -> 8.5, 16 x 8192 x 2048 70 -> 26, 64 x 8192 x 300 50 -> 12.4, 32 x 768 x 768 6.3 -> 4.8,
// 48 x 1001 x 1237 8.2 -> 5.9.
//
// An element is the sum of its wavefronts' partial sums, added in the order of the wavefronts, then of the splits;
// wavefront w of W has the steps w, w + W, ..., dealt in ascending order to four accumulators.  The short chains leave less
// error against float64 than both other kernels (3072 k: 1.2e-7 against 2.0e-7 and 5.0e-7).  B transposed and B as stored
// give the same bits, and so does a launch that may not use the memory in which the splits meet (a stream that is being
// captured): its workgroups, of sixteen wavefronts, have all splits of a tile.  Replayed with weights from memory / in cache,
// against the streaming kernel: 8 x 3072 x 768 16.9/10.4 -> 17.2/8.8 us, 1 x 8192 x 300 35/20 -> 28/18, 1 x 3072 x 768
// 14.7/5.9 -> 14.8/8.5, 1 x 16384 x 64, four tiles, 26/20 -> 29/26.  Bias, residual and the erf-form GELU follow as in the other kernels
// (tfcc/mkl/interfaces/tfcc_mklblasinterface.cpp:41-67, 69-78, 87-118).
#include <type_traits>

#include "common.hpp"
#include "sgemm_params.hpp"
#include "sgemm_skinny_plan.hpp"
#include "stream_slots.hpp"

namespace tfcc_rocm {
namespace {

using sgemm_detail::SgemmParams;
using sgemm_skinny_plan::kMaxParts;
using sgemm_skinny_plan::Plan;

typedef float skinny_v4f __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;  // two workgroups to a CU: tiles that are no multiple of the CUs even out
constexpr int kBatch = 4;  // steps asked for at once

// The memory in which the splits of a tile meet: a piece per stream, asked for by the first product that splits.
constexpr unsigned kMaxGroups = 4, kPieceTiles = kMaxParts * kMaxGroups;
struct Meeting {
  float partials[256 * (size_t)kPieceTiles];
  unsigned counts[kPieceTiles];  // zero between launches: the workgroup that arrives last sees to it
};
int clear_counts(hipStream_t stream, void* piece) {
  return tfcc_rocm_fill_async(stream, static_cast<Meeting*>(piece)->counts, 0, sizeof(unsigned), kPieceTiles);
}
StreamPieces gPieces(sizeof(Meeting), 64, clear_counts);  // 4 MB each

// TEAMS teams of eight wavefronts.  One: the workgroup has the split blockIdx.z of its tile and meets the others in `meeting`
// (null for a product that is not split).  Two, where there is no such memory: the workgroup has all splits, the teams
// taking turns; a wavefront asks for the first steps of its next split as it ends one, and the partial tiles of six splits
// wait in LDS before the workgroup meets.
//
// What is under way has to be the same on every path to a matrix op, or the compiler waits for every load before it uses the
// first (with a condition in front of every load 1 x 16384 x 64 in a graph took 37 us instead of 26): whole batches are asked for without a condition, and the last 0 to 3 steps of a wavefront have code of their own
// for each number.
template <bool TRANSB, int ROWS, int TEAMS, class Arguments>
__global__ __launch_bounds__(64 * kWaves * TEAMS, ROWS == 2 ? 2 : 4) void sgemm_skinny_kernel(const float* hotA, const float* hotB, unsigned M,
                                                                              unsigned N, unsigned K, unsigned lda, unsigned ldb,
                                                                              unsigned tilesM, unsigned tilesTotal, unsigned chunk,
                                                                              unsigned splits, unsigned perWave, Meeting* meeting,
                                                                              const Arguments arguments) {
  const SgemmParams p = arguments.whole();
  constexpr bool GROUPED = std::is_same<Arguments, SgemmParams>::value;
  constexpr unsigned ROUNDS = TEAMS == 1 ? 1 : 3, HELD = TEAMS * ROUNDS;  // splits that wait in LDS
  __shared__ float part[HELD * kWaves][4 * ROWS][64];
  __shared__ unsigned arrived;
  const unsigned lane = threadIdx.x & 63;
  const unsigned waveInGroup = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned team = TEAMS == 1 ? 0u : waveInGroup / kWaves, wave = waveInGroup - team * kWaves;
  // each XCD gets a contiguous run of tiles, the row tiles of a column tile side by side: they read the same piece of B
  const unsigned L = (blockIdx.x & 7u) * chunk + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= chunk || L >= tilesTotal) return;
  const unsigned tn = L / tilesM, tm = L - tn * tilesM, group = blockIdx.y;
  const unsigned m0 = tm * (16 * ROWS), n0 = tn * 16;
  const float* A = hotA;
  const float* B = GROUPED && p.groups ? p.groupB[group] : hotB;
  // (no range check: every offset below lies inside the operand)
  const __amdgpu_buffer_rsrc_t rsrcA = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, -1, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrcB = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), 0, -1, 0x00020000);

  // rows and columns past the edge read the last one, and their sums are dropped
  const unsigned g = lane >> 4, edge = lane & 15u;
  const unsigned col = min(n0 + edge, N - 1);
  unsigned row[ROWS], aOff[ROWS];
#pragma unroll
  for (unsigned r = 0; r < (unsigned)ROWS; ++r) {
    row[r] = min(m0 + 16 * r + edge, M - 1);
    aOff[r] = (row[r] * lda + 4 * g) * 4u;
  }
  const unsigned bOff = (TRANSB ? col * ldb + 4 * g : 4 * g * ldb + col) * 4u;
  struct Ops { float a[ROWS][4], b[4]; };
  auto load = [&](Ops& o, unsigned k) __attribute__((always_inline)) {
#pragma unroll
    for (unsigned r = 0; r < (unsigned)ROWS; ++r) {
      const auto a = __builtin_amdgcn_raw_buffer_load_b128(rsrcA, aOff[r], k * 4u, 0);
      __builtin_memcpy(o.a[r], &a, 16);
    }
    if (TRANSB) {
      const auto b = __builtin_amdgcn_raw_buffer_load_b128(rsrcB, bOff, k * 4u, 0);
      __builtin_memcpy(o.b, &b, 16);
    } else {
#pragma unroll
      for (unsigned s = 0; s < 4; ++s)
        o.b[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrcB, bOff, (k + s) * ldb * 4u, 0));
    }
  };
  const unsigned whole = K / 16, lanes = splits * kWaves;  // wavefronts that share the tile
  Ops ops[2][kBatch];
  auto loadSteps = [&](int which, unsigned step, auto steps) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < decltype(steps)::value; ++u) load(ops[which][u], (step + u * lanes) * 16u);
  };
  unsigned split = TEAMS == 1 ? blockIdx.z : team;
  unsigned first = split * kWaves + wave;

  // what the finish needs: thread t of the first 256 of every row block finishes value t / 64
  const unsigned fe = (threadIdx.x >> 6) & (4u * ROWS - 1), grow = m0 + 16 * (fe >> 2) + 4 * g + (fe & 3u), gcol = n0 + edge;
  const bool finisher = threadIdx.x < 256 * ROWS, mine = finisher && grow < M && gcol < N;
  float bv = 0.f, rv = 0.f;
  auto loadFinish = [&]() __attribute__((always_inline)) {
    const float* bias = GROUPED && p.groups ? p.groupBias[group] : p.bias;
    if (mine && bias) bv = bias[gcol];
    if (mine && p.residual) rv = p.residual[(size_t)grow * N + gcol];
  };

  skinny_v4f acc[ROWS][kBatch];  // one for each step of a batch: short chains, for the rounding and for the matrix ops' latency
  auto multiply = [&](const Ops& o, int u) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int r = 0; r < ROWS; ++r) acc[r][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[r][s], o.b[s], acc[r][u], 0, 0, 0);
  };
  auto multiplySteps = [&](int which, auto steps) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < decltype(steps)::value; ++u) multiply(ops[which][u], u);
  };
  const std::integral_constant<int, kBatch> batch;
  auto with = [](unsigned steps, auto f) __attribute__((always_inline)) {  // 0 to 3
    if (steps < 2) {
      if (steps == 0) f(std::integral_constant<int, 0>{});
      else f(std::integral_constant<int, 1>{});
    } else {
      if (steps == 2) f(std::integral_constant<int, 2>{});
      else f(std::integral_constant<int, 3>{});
    }
  };
  // The wavefront's steps of its split: first, first + lanes, ...; perWave of them, or one more.  Whoever shares a tile has
  // at least four, and a first batch that has been asked for.
  const unsigned oneMore = whole - perWave * lanes;
  auto sumSplit = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kBatch * ROWS; ++u) acc[u / kBatch][u % kBatch] = skinny_v4f{0.f, 0.f, 0.f, 0.f};
    const unsigned steps = perWave + (first < oneMore ? 1u : 0u);
    if (TEAMS == 1 && steps < kBatch) {
      with(steps, [&](auto few) {
        loadSteps(0, first, few);
        if (TEAMS == 1) loadFinish();
        multiplySteps(0, few);
      });
      return;
    }
    loadSteps(0, first, batch);
    unsigned left = steps - kBatch, next = first + kBatch * lanes;  // what has not been asked for
    for (; left >= 2 * kBatch; left -= 2 * kBatch, next += 2 * kBatch * lanes) {
      loadSteps(1, next, batch);
      multiplySteps(0, batch);
      loadSteps(0, next + kBatch * lanes, batch);
      multiplySteps(1, batch);
    }
    if (left >= kBatch) {
      loadSteps(1, next, batch);
      multiplySteps(0, batch);
      with(left - kBatch, [&](auto few) {
        loadSteps(0, next + kBatch * lanes, few);
        if (TEAMS == 1) loadFinish();
        multiplySteps(1, batch);
        multiplySteps(0, few);
      });
    } else {
      with(left, [&](auto few) {
        loadSteps(1, next, few);
        if (TEAMS == 1) loadFinish();
        multiplySteps(0, batch);
        multiplySteps(1, few);
      });
    }
  };
  auto keepSplit = [&](unsigned held) __attribute__((always_inline)) {
    if (K % 16 != 0 && first == whole % lanes) {  // the step in which K ends
      Ops o;
#pragma unroll
      for (unsigned s = 0; s < 4; ++s) {
        const bool in = whole * 16 + 4 * g + s < K;
#pragma unroll
        for (unsigned r = 0; r < (unsigned)ROWS; ++r) o.a[r][s] = in ? A[(size_t)row[r] * lda + whole * 16 + 4 * g + s] : 0.f;
        const size_t k = whole * 16 + 4 * g + s;
        o.b[s] = in ? B[TRANSB ? (size_t)col * ldb + k : k * ldb + col] : 0.f;
      }
      multiply(o, 0);
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part[held * kWaves + wave][4 * r + e][lane] = (acc[r][0][e] + acc[r][1][e]) + (acc[r][2][e] + acc[r][3][e]);
  };
  float v = 0.f;
  auto meet = [&](unsigned from, unsigned to) __attribute__((always_inline)) {  // adds the held splits from .. to - 1
    __syncthreads();
    if (!finisher) return;
    for (unsigned s = from; s < to; ++s) {
      float sum = part[(s - from) * kWaves][fe][lane];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) sum += part[(s - from) * kWaves + w][fe][lane];
      v = s == 0 || TEAMS == 1 ? sum : v + sum;
    }
  };
  if constexpr (TEAMS == 1) {
    sumSplit();
    keepSplit(0);
    meet(split, split + 1);
  } else {
    unsigned met = 0;
    for (;;) {
      if (split < splits) {
        sumSplit();
        if (met == 0 && split == team) loadFinish();
        keepSplit(split - met);
      }
      split += TEAMS;
      first += TEAMS * kWaves;
      const unsigned through = split - team;  // every split below it has been summed
      if (through >= splits || through - met == HELD) {  // the same for the whole workgroup
        const unsigned to = min(through, splits);
        meet(met, to);
        met = to;
        if (met == splits) break;
        __syncthreads();
      }
    }
  }

  if (TEAMS == 1 && splits > 1) {
    // The partial tile goes past the caches, and waiting for the store is all the order there has to be in front of the
    // count; the workgroup that arrives last adds the partial tiles in the order of the splits.
    const unsigned tile = group * tilesTotal + L;
    float* mineAt = meeting->partials + (size_t)tile * splits * (256 * ROWS);
    unsigned* count = meeting->counts + tile;
    if (finisher) __hip_atomic_store(mineAt + blockIdx.z * (256 * ROWS) + threadIdx.x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) arrived = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != splits - 1) return;
    if (threadIdx.x == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (finisher) {
      v = __hip_atomic_load(mineAt + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (unsigned s = 1; s < splits; ++s)
        v += __hip_atomic_load(mineAt + s * (256 * ROWS) + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (!mine) return;
  v += bv;
  if (p.residual) v += rv;
  if (p.act == 1) v = gelu_erf_f32(v);
  float* C = GROUPED && p.groups ? p.groupC[group] : p.C;
  C[(size_t)grow * p.ldc + gcol] = v;
}

template <bool TRANSB>
int launch_skinny(hipStream_t stream, SgemmParams p, const Plan& plan) {
  const unsigned groups = p.groups ? p.groups : 1u;
  p.batch = 1;
  const unsigned splits = plan.splits;
  Meeting* meeting = nullptr;
  if (splits > 1) {
    int dev = 0;
    TFCC_HIP_CHECK(hipGetDevice(&dev));
    meeting = static_cast<Meeting*>(gPieces.of(dev, stream));
  }
  // (The same bits with one row block as with two.)
  const bool alone = splits > 1 && meeting == nullptr, two = plan.rows == 2 && !alone;
  if (!sgemm_detail::set_tiles(p, two ? 32 : 16, 16)) return set_error(TFCC_ROCM_INVALID_ARGUMENT, "sgemm: too many tiles");
  auto launch = [&](const auto& arguments) {
    using Arguments = std::decay_t<decltype(arguments)>;
    auto kern = alone ? sgemm_skinny_kernel<TRANSB, 1, 2, Arguments>
                : two ? sgemm_skinny_kernel<TRANSB, 2, 1, Arguments>
                      : sgemm_skinny_kernel<TRANSB, 1, 1, Arguments>;
    hipLaunchKernelGGL(kern, dim3(p.chunk * 8, groups, alone ? 1u : splits), dim3(64 * kWaves * (alone ? 2 : 1)), 0, stream, p.A, p.B,
                       (unsigned)p.M, (unsigned)p.N, (unsigned)p.K, (unsigned)p.lda, (unsigned)p.ldb, p.tilesM, p.tilesTotal, p.chunk,
                       splits, p.K / 16 / (splits * kWaves), meeting, arguments);
  };
  if (p.groups) launch(p);
  else launch(sgemm_detail::SgemmFinish(p));
  return check_launch("sgemm");
}

}  // namespace

namespace sgemm_detail {

int sgemm_skinny_launch(hipStream_t stream, const SgemmParams& p, const Plan& plan, bool transB) {
  return transB ? launch_skinny<true>(stream, p, plan) : launch_skinny<false>(stream, p, plan);
}

void sgemm_skinny_release_stream(int dev, hipStream_t stream) { gPieces.release(dev, stream); }

}  // namespace sgemm_detail
}  // namespace tfcc_rocm
