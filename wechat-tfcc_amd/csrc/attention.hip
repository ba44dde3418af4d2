// softmax(Q K^T [/ divisor]) V per batch entry in one launch: key sequences of up to 128 rows with the scores of a
// row block in LDS in one piece (attention_kernel), and longer ones in runs of 32 keys (attention_stream_kernel).
//
// Stands where the reference's runtime runs the attention core of an encoder layer as separate
// operations on tensors in HBM: Matmul (tfcc_runtime/operations/math/matmul.cpp:27-41), Div by a
// value, Softmax (tfcc_runtime/operations/math/softmax.cpp), Matmul again, with base::transpose
// (tfcc/core/operations/tfcc_base.cpp:124-134) before and after.  Here the score matrix of a block of
// 64 query rows never leaves the CU: Q is held in registers, K in LDS, the scores and probabilities in
// LDS, V in registers until the scores are done and then in K's place (70.7 KB, two workgroups per CU).
//
// Every number is computed by the same instruction sequence as in the three separate kernels
// (fp32 32x32x2 matrix ops over ascending k into one accumulator; the softmax of one row by one
// wavefront holding columns l and l + 64), and is rounded to fp32 between the steps, so the result
// equals theirs bit for bit.
#include <float.h>

#include "attention_plan.hpp"
#include "common.hpp"
#include "qgemm_params.hpp"  // UDiv: division by multiply-high

namespace tfcc_rocm {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kRows = 64;        // query rows per workgroup
constexpr int kMaxT = attention_plan::kWholeKeys;  // key rows
constexpr int kMaxD = 64;        // head width
constexpr int kPitchK = kMaxD + 4;    // floats; 128-bit row reads of 32 consecutive rows hit all banks once
constexpr int kPitchV = kMaxD + 8;    // 32-bit reads of rows r and r + 4 land 32 banks apart
constexpr int kPitchS = kMaxT + 4;
// K and, once the scores are done, V share one region; Q stays in registers.  70.7 KB: two workgroups per CU.
constexpr int kLdsFloats = kMaxT * kPitchV + kRows * kPitchS;

struct AttentionParams {
  const float* Q;
  const float* K;
  const float* V;
  float* O;
  unsigned S, T, D;
  unsigned ldq, ldk, ldv, ldo;
  unsigned long long outerQ, outerK, outerV, outerO;
  unsigned long long innerQ, innerK, innerV, innerO;
  unsigned batchInner, blocksS, total, chunk;
  float divisor;
  int divide;
  const float* mask;  // optional: one value per key column, added to the (divided) scores of every query row
  unsigned long long outerM, innerM;
  unsigned blocksMagic, blocksShift, innerMagic, innerShift;  // division by blocksS and by batchInner as multiply-high
};

// Everything the kernels read of the argument block, named before the first branch: one round trip to memory for it
// instead of one per basic block, at the head of a launch of ten to twenty microseconds.
#define TFCC_ATTENTION_FETCH_ARGUMENTS(p)                                                                              \
  asm volatile("" ::"s"(p.Q), "s"(p.K), "s"(p.V), "s"(p.O), "s"(p.S), "s"(p.T), "s"(p.D), "s"(p.ldq), "s"(p.ldk),      \
               "s"(p.ldv), "s"(p.ldo), "s"(p.outerQ), "s"(p.outerK), "s"(p.outerV), "s"(p.outerO), "s"(p.innerQ),      \
               "s"(p.innerK), "s"(p.innerV), "s"(p.innerO), "s"(p.batchInner), "s"(p.blocksS), "s"(p.total),           \
               "s"(p.chunk), "s"(p.divisor), "s"(p.divide), "s"(p.mask), "s"(p.outerM), "s"(p.innerM),                 \
               "s"(p.blocksMagic), "s"(p.blocksShift), "s"(p.innerMagic), "s"(p.innerShift))


// ROWS query rows per workgroup, a wavefront per eight of them: 64 rows (eight wavefronts, 70.7 KB, two workgroups per
// CU) when every CU gets at most one workgroup that way, 32 rows (four wavefronts, 53.8 KB, three per CU) when the
// 64-row blocks would pile up two on some CUs and one or none on others (16 x 12 heads of 128 rows: 384 blocks of 64
// on 256 CUs against 768 blocks of 32, three on every CU).  The arithmetic per element is the same.
template <int ROWS>
__global__ __launch_bounds__(8 * ROWS, ROWS == 64 ? 4 : 3) void attention_kernel(const AttentionParams p) {
  constexpr int kRows = ROWS, kThreads = 8 * ROWS;
  static_assert(ROWS == 64 || ROWS == 32, "two or one row blocks of 32");
  extern __shared__ __align__(16) float lds[];
  float* KVs = lds;                       // K as [128][kPitchK], later V as [128][kPitchV]
  float* Sc = KVs + kMaxT * kPitchV;      // [64][kPitchS]  scores, then probabilities

  // consecutive workgroup ids land on different XCDs: the blocks of one head stay on one XCD
  const unsigned wg = blockIdx.x;
  TFCC_ATTENTION_FETCH_ARGUMENTS(p);
  const unsigned L = (wg & 7u) * p.chunk + (wg >> 3);
  if ((wg >> 3) >= p.chunk || L >= p.total) return;
  const unsigned bi = udiv_apply(L, p.blocksMagic, p.blocksShift), blk = L - bi * p.blocksS;
  const unsigned bo = udiv_apply(bi, p.innerMagic, p.innerShift), bn = bi - bo * p.batchInner;
  const unsigned s0 = blk * kRows;
  const unsigned S = p.S, T = p.T, D = p.D;
  const float* __restrict__ Q = p.Q + (size_t)bo * p.outerQ + (size_t)bn * p.innerQ;
  const float* __restrict__ K = p.K + (size_t)bo * p.outerK + (size_t)bn * p.innerK;
  const float* __restrict__ V = p.V + (size_t)bo * p.outerV + (size_t)bn * p.innerV;
  float* __restrict__ O = p.O + (size_t)bo * p.outerO + (size_t)bn * p.innerO;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // this lane's two mask values, fetched now: the softmax phase that adds them is far away
  const bool masked = p.mask != nullptr;
  float mk[2] = {0.f, 0.f};
  if (masked) {
    const float* __restrict__ mrow = p.mask + (size_t)bo * p.outerM + (size_t)bn * p.innerM;
#pragma unroll
    for (int q = 0; q < 2; ++q)
      if ((unsigned)lane + 64u * q < T) mk[q] = mrow[lane + 64 * q];
  }
  const int lrow = lane & 31, g = lane >> 5;
  const unsigned Dp = (D + 7u) & ~7u;   // k extent of the score product
  const unsigned Tp = (T + 7u) & ~7u;   // k extent of the second product

  // ---- loads.  K goes to LDS; Q goes through the region the scores will later occupy into the registers
  // the score product takes it from; V waits in registers until K is no longer needed.  A buffer load whose
  // offset lies past the end of its operand returns zero: that is how everything past the operands' extents
  // that a matrix op will read becomes zero.
  const int wmS = wave >> 2, wnS = wave & 3;  // scores: ROWS / 32 x 4 wavefronts, one 32 x 32 block each
  constexpr int CH = kMaxD / 4;               // 16-byte chunks per row
  constexpr int KV_ITEMS = kMaxT * CH / kThreads, Q_ITEMS = kRows * CH / kThreads, KBQ = kMaxD / 8;
  constexpr unsigned kPastEnd = 0xfffffff0u;
  v4f qf[KBQ], vreg[KV_ITEMS];
  {
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(Q), 0, (int)(((S - 1) * p.ldq + D) * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(K), 0, (int)(((T - 1) * p.ldk + D) * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(V), 0, (int)(((T - 1) * p.ldv + D) * 4u), 0x00020000);
    v4f qreg[Q_ITEMS], kreg[KV_ITEMS];
#pragma unroll
    for (int it = 0; it < Q_ITEMS; ++it) {
      const unsigned w = tid + it * kThreads, row = s0 + w / CH, ch = w % CH;
      qreg[it] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                             rq, (row < S && ch * 4 < D) ? (row * p.ldq + ch * 4) * 4u : kPastEnd, 0, 0));
    }
#pragma unroll
    for (int it = 0; it < KV_ITEMS; ++it) {
      const unsigned w = tid + it * kThreads, row = w / CH, ch = w % CH;
      const bool in = row < T && ch * 4 < D;
      kreg[it] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rk, in ? (row * p.ldk + ch * 4) * 4u : kPastEnd, 0, 0));
      vreg[it] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rv, in ? (row * p.ldv + ch * 4) * 4u : kPastEnd, 0, 0));
    }
#pragma unroll
    for (int it = 0; it < KV_ITEMS; ++it) {
      const int w = tid + it * kThreads, row = w / CH, ch = w % CH;
      *reinterpret_cast<v4f*>(KVs + row * kPitchK + ch * 4) = kreg[it];
    }
#pragma unroll
    for (int it = 0; it < Q_ITEMS; ++it) {
      const int w = tid + it * kThreads, row = w / CH, ch = w % CH;
      *reinterpret_cast<v4f*>(Sc + row * kPitchK + ch * 4) = qreg[it];
    }
  }
  __syncthreads();
  {
    const float* qa = Sc + (32 * wmS + lrow) * kPitchK + 4 * g;
#pragma unroll
    for (int kb = 0; kb < KBQ; ++kb) {
      qf[kb] = v4f{0.f, 0.f, 0.f, 0.f};
      if ((unsigned)kb * 8 < Dp) qf[kb] = *reinterpret_cast<const v4f*>(qa + kb * 8);
    }
  }

  // ---- scores.  All K operands are fetched from LDS before the first matrix op, so that their latency
  // is paid once.  A divisor that is a power of two divides exactly like a multiplication by its reciprocal.
  const bool liveS = (unsigned)(32 * wnS) < T;  // wave-uniform: this wavefront's 32 columns exist
  v4f bf[KBQ];
  {
    const float* ka = KVs + (32 * wnS + lrow) * kPitchK + 4 * g;
#pragma unroll
    for (int kb = 0; kb < KBQ; ++kb) {
      bf[kb] = v4f{0.f, 0.f, 0.f, 0.f};
      if (liveS && (unsigned)kb * 8 < Dp) bf[kb] = *reinterpret_cast<const v4f*>(ka + kb * 8);
    }
  }
  __syncthreads();  // every wavefront has taken its Q operands out of the region the scores go to
  if (liveS) {
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int kb = 0; kb < KBQ; ++kb) {
      if ((unsigned)kb * 8 < Dp) {
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(qf[kb][s], bf[kb][s], acc, 0, 0, 0);
      }
    }
    float* sc = Sc + (32 * wmS + 4 * g) * kPitchS + 32 * wnS + lrow;
    const float divisor = p.divisor;
    const unsigned bits = __builtin_bit_cast(unsigned, divisor), expo = (bits >> 23) & 0xffu;
    if (!p.divide) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[(8 * (r / 4) + (r & 3)) * kPitchS] = acc[r];
    } else if ((bits & 0x007fffffu) == 0 && expo >= 2 && expo <= 252) {
      const float inverse = 1.0f / divisor;  // exact: also a power of two
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[(8 * (r / 4) + (r & 3)) * kPitchS] = acc[r] * inverse;
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[(8 * (r / 4) + (r & 3)) * kPitchS] = acc[r] / divisor;
    }
  }
  __syncthreads();

  // ---- K is done with: V takes its place
#pragma unroll
  for (int it = 0; it < KV_ITEMS; ++it) {
    const int w = tid + it * kThreads, row = w / CH, ch = w % CH;
    *reinterpret_cast<v4f*>(KVs + row * kPitchV + ch * 4) = vreg[it];
  }

  // ---- softmax of each row by one wavefront, eight rows in flight; columns T .. Tp-1 become the zeros
  // the next product reads
  {
    const unsigned rows = min((unsigned)kRows, S - s0);
    constexpr int R = 8, W = kThreads / 64;  // R is the eight of wave_reduce8
    for (unsigned base = wave; base < rows; base += W * R) {
      float v[R][2], mx[R], sum[R];
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const unsigned row = min(base + W * u, (unsigned)kRows - 1);  // a row past the block's end is computed and dropped
        const float* sc = Sc + row * kPitchS;
        mx[u] = -FLT_MAX;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const unsigned i = lane + 64 * q;
          v[u][q] = i < T ? (masked ? sc[i] + mk[q] : sc[i]) : -FLT_MAX;
          mx[u] = fmaxf(mx[u], v[u][q]);
        }
      }
      wave_reduce8<true>(mx, lane);
#pragma unroll
      for (int u = 0; u < R; ++u) {
        sum[u] = 0.f;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const unsigned i = lane + 64 * q;
          v[u][q] = i < T ? softmax_exp(v[u][q] - mx[u]) : 0.f;
          sum[u] += v[u][q];
        }
      }
      wave_reduce8<false>(sum, lane);
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const unsigned row = base + W * u;
        if (row < rows) {
          float* sc = Sc + row * kPitchS;
          const float inverse = 1.0f / sum[u];  // as the stand-alone softmax: one division per row
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const unsigned i = lane + 64 * q;
            sc[i] = i < T ? v[u][q] * inverse : 0.f;
          }
        }
      }
    }
  }
  __syncthreads();

  if constexpr (ROWS == 64) {
    // ---- probabilities x V: the first four wavefronts, (wm, wn) owning rows 32*wm.. and columns 32*wn.. of the
    // 64 x D result (one accumulator per element over all of T, as in a product of its own)
    const int wm = wave >> 1, wn = wave & 1;
    if (wave < 4 && (unsigned)(32 * wn) < D) {
      constexpr int KB = kMaxT / 8, HALF = KB / 2;
      v16f acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
      const float* pa = Sc + (32 * wm + lrow) * kPitchS + 4 * g;
      const float* vb = KVs + (4 * g) * kPitchV + 32 * wn + lrow;
#pragma unroll
      for (int h = 0; h < 2; ++h) {  // operands are fetched from LDS for eight steps at a time
        v4f af[HALF], bf[HALF];
#pragma unroll
        for (int q = 0; q < HALF; ++q) {
          const int kb = h * HALF + q;
          af[q] = v4f{0.f, 0.f, 0.f, 0.f};
          bf[q] = v4f{0.f, 0.f, 0.f, 0.f};
          if ((unsigned)kb * 8 < Tp) {
            af[q] = *reinterpret_cast<const v4f*>(pa + kb * 8);
#pragma unroll
            for (int s = 0; s < 4; ++s) bf[q][s] = vb[(kb * 8 + s) * kPitchV];
          }
        }
#pragma unroll
        for (int q = 0; q < HALF; ++q) {
          if ((unsigned)(h * HALF + q) * 8 < Tp) {
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(af[q][s], bf[q][s], acc, 0, 0, 0);
          }
        }
      }
      const unsigned col = 32 * wn + lrow;
      if (s0 + 32 * wm + 32 <= S && 32u * wn + 32 <= D && p.ldo < (1u << 24)) {
        // a whole 32 x 32 block: a register per lane (row 4g, column lrow), a scalar per row, no checks
        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
            O + (size_t)(s0 + 32 * wm) * p.ldo + 32 * wn, 0, 0x7fffffff, 0x00020000);
        const unsigned voff = ((4 * g) * p.ldo + lrow) * 4u;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float value = acc[r];  // a copy: __builtin_bit_cast applied to a vector element reads element 0
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, value), ro, voff,
                                                (8 * (r / 4) + (r & 3)) * p.ldo * 4u, 0);
        }
      } else if (col < D) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const unsigned row = s0 + 32 * wm + 8 * (r / 4) + 4 * g + (r & 3);
          if (row < S) O[(size_t)row * p.ldo + col] = acc[r];
        }
      }
    }
  } else {
    // ---- probabilities x V.  A product of its own sums each element in one accumulator over k in the order
    // 8kb + s, 8kb + 4 + s (s = 0..3) with 32x32x2 matrix ops; the 16x16x4 op adds its four k values to the accumulator
    // one after the other in lane-group order, so feeding lane groups 0..3 the k values 8kb + 2h, 8kb + 4 + 2h,
    // 8kb + 2h + 1, 8kb + 5 + 2h in ops h = 0, 1 gives the same bits - and blocks of 16 x 16 divide the ROWS x D
    // result evenly among all wavefronts: wavefront w owns rows 16 (w / 2).. and the column blocks 2 (w & 1), 2 (w & 1) + 1.
  // With 32 rows this keeps all four SIMDs busy (two 32 x 32 blocks would occupy two); with 64 rows it measured a
  // microsecond slower than the four 32 x 32 blocks above (twice the LDS operand reads, two-way bank conflicts).
    {
      constexpr int KB = kMaxT / 8;
      const int l16 = lane & 15, q = lane >> 4;
      const int rb = wave >> 1, cb0 = 2 * (wave & 1);
      const int kq = (q >> 1) + 4 * (q & 1);  // this lane group's k inside a block of eight, op 0 (op 1: + 2)
      const float* pa = Sc + (16 * rb + l16) * kPitchS + kq;
      const float* vb = KVs + kq * kPitchV + 16 * cb0 + l16;
      const bool live[2] = {(unsigned)(16 * cb0) < D, (unsigned)(16 * cb0 + 16) < D};
      v4f acc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
      if (live[0]) {
        float af[KB][2], bf[2][KB][2];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            af[kb][h] = 0.f; bf[0][kb][h] = 0.f; bf[1][kb][h] = 0.f;
          }
          if ((unsigned)kb * 8 < Tp) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              af[kb][h] = pa[kb * 8 + 2 * h];
              bf[0][kb][h] = vb[(kb * 8 + 2 * h) * kPitchV];
              bf[1][kb][h] = vb[(kb * 8 + 2 * h) * kPitchV + 16];  // columns past D hold zeros
            }
          }
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          if ((unsigned)kb * 8 < Tp) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[kb][h], bf[0][kb][h], acc[0], 0, 0, 0);
              acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[kb][h], bf[1][kb][h], acc[1], 0, 0, 0);
            }
          }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (!live[j]) continue;
          const unsigned c0 = 16 * (cb0 + j), r0 = s0 + 16 * rb;
          if (r0 + 16 <= S && c0 + 16 <= D && p.ldo < (1u << 24)) {
            // a whole 16 x 16 block: a register per lane (row 4q, column l16), a scalar per row, no checks
            const __amdgpu_buffer_rsrc_t ro =
                __builtin_amdgcn_make_buffer_rsrc(O + (size_t)r0 * p.ldo + c0, 0, 0x7fffffff, 0x00020000);
            const unsigned voff = ((4 * q) * p.ldo + l16) * 4u;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float value = acc[j][r];  // a copy: __builtin_bit_cast applied to a vector element reads element 0
              __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, value), ro, voff, r * p.ldo * 4u, 0);
            }
          } else if (c0 + l16 < D) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const unsigned row = r0 + 4 * q + r;
              if (row < S) O[(size_t)row * p.ldo + c0 + l16] = acc[j][r];
            }
          }
        }
      }
    }
  }
}

// The same with 16 query rows per workgroup of four wavefronts, bound by the chain from the first load to the last store, of
// which every part is half as long here, rather than by a rate.  No operand goes
// through LDS on its way in: the 16x16x4 ops take k as 0, 4, 1, 5 and 2, 6, 3, 7 of every eight (above), so of two blocks of
// eight each half of a wavefront fetches one, four values to a load, and one exchange between the halves makes the operands
// of two ops.  The scores are the first thing that the wavefronts share.  KEYS: 64 or 128, one or two columns of the softmax
// to a lane.  12 heads of 64 columns, us, 32 or 64 rows -> 16: 1 x 16 rows 6.2 -> 4.0, 1 x 29 6.7 -> 4.1, 1 x 64 6.9 -> 4.5, 1 x
// 128 7.9 -> 6.1, 8 x 29 6.8 -> 4.3, 16 x 64 9.0 -> 8.0, 64 x 64 22.0 -> 20.2.
__device__ __forceinline__ void operands16(const v4f& x, float (&op)[2][2]) {  // [block of eight][op]
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float low = x[2 * h], high = x[2 * h + 1];  // copies: a bit_cast of a vector's element reads its first one
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, low), __builtin_bit_cast(unsigned, high), false, false);
    op[0][h] = __builtin_bit_cast(float, (unsigned)r[0]);
    op[1][h] = __builtin_bit_cast(float, (unsigned)r[1]);
  }
}

template <int KEYS>
__global__ __launch_bounds__(256, 1) void attention_rows16_kernel(const AttentionParams p) {
  static_assert(KEYS == 64 || KEYS == 128, "one or two columns to a lane");
  constexpr int ROWS = 16, PER = KEYS / 64, PAIRS_D = kMaxD / 16, PAIRS_T = KEYS / 16, PITCH = KEYS + 4;
  __shared__ __attribute__((aligned(16))) float Sc[ROWS * PITCH];  // scores, then probabilities
  const unsigned wg = blockIdx.x;
  TFCC_ATTENTION_FETCH_ARGUMENTS(p);
  const unsigned L = (wg & 7u) * p.chunk + (wg >> 3);
  if ((wg >> 3) >= p.chunk || L >= p.total) return;
  const unsigned bi = udiv_apply(L, p.blocksMagic, p.blocksShift), blk = L - bi * p.blocksS;
  const unsigned bo = udiv_apply(bi, p.innerMagic, p.innerShift), bn = bi - bo * p.batchInner;
  const unsigned s0 = blk * ROWS, S = p.S, T = p.T, D = p.D;
  const float* __restrict__ Q = p.Q + (size_t)bo * p.outerQ + (size_t)bn * p.innerQ;
  const float* __restrict__ K = p.K + (size_t)bo * p.outerK + (size_t)bn * p.innerK;
  const float* __restrict__ V = p.V + (size_t)bo * p.outerV + (size_t)bn * p.innerV;
  float* __restrict__ O = p.O + (size_t)bo * p.outerO + (size_t)bn * p.innerO;
  const unsigned lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned Dp = (D + 7u) & ~7u, Tp = (T + 7u) & ~7u;

  // ---- loads, in the order of their use; an offset past the end of its operand returns zero
  constexpr unsigned kPastEnd = 0xfffffff0u;
  auto buffer = [&](const float* x, unsigned rows, unsigned ld) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0, (int)(((rows - 1) * ld + D) * 4u), 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rq = buffer(Q, S, p.ldq), rk = buffer(K, T, p.ldk), rv = buffer(V, T, p.ldv);
  const unsigned chunk = 2 * (q >> 1) + (q & 1);  // of four values, in a pair of blocks of eight
  auto load_row = [&](__amdgpu_buffer_rsrc_t from, unsigned row, unsigned rows, unsigned ld, v4f (&x)[PAIRS_D]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PAIRS_D; ++j) {
      const unsigned at = 16 * j + 4 * chunk;
      x[j] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(from, row < rows && at < D ? (row * ld + at) * 4u : kPastEnd, 0, 0));
    }
  };
  v4f qreg[PAIRS_D], kreg[PER][PAIRS_D];
  load_row(rq, s0 + l16, S, p.ldq, qreg);
#pragma unroll
  for (int b = 0; b < PER; ++b) load_row(rk, 16 * (wave + 4 * b) + l16, T, p.ldk, kreg[b]);
  const bool masked = p.mask != nullptr;
  float mk[PER] = {};
  if (masked) {
    const float* __restrict__ mrow = p.mask + (size_t)bo * p.outerM + (size_t)bn * p.innerM;
#pragma unroll
    for (int c = 0; c < PER; ++c)
      if (lane + 64u * c < T) mk[c] = mrow[lane + 64 * c];
  }
  const unsigned kq = (q >> 1) + 4 * (q & 1), col = 16 * wave + l16;
  float vreg[2 * PAIRS_T][2];
#pragma unroll
  for (int kb = 0; kb < 2 * PAIRS_T; ++kb)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned row = 8 * kb + kq + 2 * h;
      vreg[kb][h] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, row < T && col < D ? (row * p.ldv + col) * 4u : kPastEnd, 0, 0));
    }

  // ---- scores: wavefront w has the columns 16w .. and 64 + 16w ..
  {
    v4f acc[PER];
#pragma unroll
    for (int b = 0; b < PER; ++b) acc[b] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < PAIRS_D; ++j) {
      float qo[2][2], ko[PER][2][2];
      operands16(qreg[j], qo);
#pragma unroll
      for (int b = 0; b < PER; ++b) operands16(kreg[b][j], ko[b]);
#pragma unroll
      for (int e = 0; e < 2; ++e)
        if ((unsigned)(16 * j + 8 * e) < Dp) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int b = 0; b < PER; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(qo[e][h], ko[b][e][h], acc[b], 0, 0, 0);
        }
    }
    // a divisor that is a power of two divides exactly like a multiplication by its reciprocal
    const float divisor = p.divisor;
    const unsigned bits = __builtin_bit_cast(unsigned, divisor), expo = (bits >> 23) & 0xffu;
    const bool exact = (bits & 0x007fffffu) == 0 && expo >= 2 && expo <= 252;
    const float inverse = exact ? 1.0f / divisor : 0.f;
#pragma unroll
    for (int b = 0; b < PER; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        Sc[(4 * q + r) * PITCH + 16 * (wave + 4 * b) + l16] = !p.divide ? acc[b][r] : exact ? acc[b][r] * inverse : acc[b][r] / divisor;
  }
  __syncthreads();

  // ---- softmax: four rows by a wavefront; columns T .. become the zeros the next product reads
  {
    float v[4][PER], mx[4], sum[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      mx[u] = -FLT_MAX;
#pragma unroll
      for (int c = 0; c < PER; ++c) {
        const unsigned i = lane + 64 * c;
        const float score = Sc[(wave + 4 * u) * PITCH + i];
        v[u][c] = i < T ? (masked ? score + mk[c] : score) : -FLT_MAX;
        mx[u] = fmaxf(mx[u], v[u][c]);
      }
    }
    wave_reduce4<true>(mx);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      sum[u] = 0.f;
#pragma unroll
      for (int c = 0; c < PER; ++c) {
        v[u][c] = lane + 64 * c < T ? softmax_exp(v[u][c] - mx[u]) : 0.f;
        sum[u] += v[u][c];
      }
    }
    wave_reduce4<false>(sum);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float inverse = 1.0f / sum[u];  // as the stand-alone softmax: one division per row
#pragma unroll
      for (int c = 0; c < PER; ++c) Sc[(wave + 4 * u) * PITCH + lane + 64 * c] = lane + 64 * c < T ? v[u][c] * inverse : 0.f;
    }
  }
  __syncthreads();

  // ---- probabilities x V: wavefront w has the columns 16w ..
  if (16 * wave >= D) return;
  v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < PAIRS_T; ++j) {
    if ((unsigned)(16 * j) >= Tp) break;
    float po[2][2];
    operands16(*reinterpret_cast<const v4f*>(&Sc[l16 * PITCH + 16 * j + 4 * chunk]), po);
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if ((unsigned)(16 * j + 8 * e) < Tp) {
#pragma unroll
        for (int h = 0; h < 2; ++h) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(po[e][h], vreg[2 * j + e][h], acc, 0, 0, 0);
      }
  }
  if (col < D) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned row = s0 + 4 * q + r;
      if (row < S) O[(size_t)row * p.ldo + col] = acc[r];
    }
  }
}

// ---- the same for key sequences of any length: each of four wavefronts takes every fourth run of 32 keys, with a maximum, a sum
// and a result of its own for every query row (m, l, o).  Per run: scores; p = exp(score - m_new) with m_new = max(m, the run's
// maximum); l and o scaled by exp(m - m_new), then the run's p and p V added.  At the end the wavefronts' l and o meet, scaled by
// exp(m - the largest m), and every row is divided by its l.  The same real function as the three separate kernels, summed in a
// different order: results agree with them to a few units in the last place, not bit for bit; the contract checked is
// the relative error against double precision.
//
// Nothing goes through LDS before the end, and no wavefront waits for another.  The scores are formed transposed, keys x queries:
// lane (l16, q) of a 16 x 16 block then holds keys 4q .. 4q + 3 of query l16, which is what the ops of the second product,
// V^T p^T, take from it as they stand, and m, l and the scale belong to the lane's own query.  Which k an op's four lane groups
// have is the same choice for both operands, so K, Q and V are fetched four values to a load: row l16 of Q and K from 4q on,
// and of V's row of a key columns 4 l16 .. + 3, whose e-th values make one block of results (row i of it is column 4i + e).
// BLOCKS: of 16 query rows, which share the loads of K and V.
//
// Few blocks: bound by the chain of a wavefront's runs; many: by the matrix ops (16 x 12 heads of 512 keys: 82 of 131 us) and the vector
// work between them.  Loads take no vector instruction (a descriptor begins at the run's first key and the offsets stay), and keys
// past the last one are looked for in the last run alone: 16 x 12 x 512 157 -> 131.  12 heads of 64 columns, us, workgroups of 32 or 64
// rows walking blocks of 128 keys through LDS -> this: 1 x 160 14.4 -> 6.3, 1 x 384 22.7 -> 12.7, 4 x 256 19.1 -> 14.4, 4 x 384 51 ->
// 27, 16 x 512 200 -> 131; error against float64 4.0e-7 -> 3.2e-7 with 256 keys, 8.7e-7 -> 5.1e-7 with 2048.
template <int BLOCKS>
__global__ __launch_bounds__(256, 2) void attention_stream_kernel(const AttentionParams p) {
  constexpr int WAVES = 4, ROWS = 16 * BLOCKS, QUADS = kMaxD / 16, GROUPS = 2, RUN = 16 * GROUPS;
  static_assert(QUADS == 4 && WAVES == 4, "a wavefront finishes one of four quads of columns");
  __shared__ v4f part[WAVES][BLOCKS][4][64];
  __shared__ float wm[WAVES][ROWS], wl[WAVES][ROWS];
  const unsigned wg = blockIdx.x;
  TFCC_ATTENTION_FETCH_ARGUMENTS(p);
  const unsigned L = (wg & 7u) * p.chunk + (wg >> 3);
  if ((wg >> 3) >= p.chunk || L >= p.total) return;
  const unsigned bi = udiv_apply(L, p.blocksMagic, p.blocksShift), blk = L - bi * p.blocksS;
  const unsigned bo = udiv_apply(bi, p.innerMagic, p.innerShift), bn = bi - bo * p.batchInner;
  const unsigned s0 = blk * ROWS, S = p.S, T = p.T, D = p.D;
  const float* __restrict__ Q = p.Q + (size_t)bo * p.outerQ + (size_t)bn * p.innerQ;
  const float* __restrict__ K = p.K + (size_t)bo * p.outerK + (size_t)bn * p.innerK;
  const float* __restrict__ V = p.V + (size_t)bo * p.outerV + (size_t)bn * p.innerV;
  float* __restrict__ O = p.O + (size_t)bo * p.outerO + (size_t)bn * p.innerO;
  const unsigned lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // An offset past the end of its operand returns zero; the operand begins at the run's first key, so the offsets stay.
  constexpr unsigned kPastEnd = 0xfffffff0u;
  auto rows_from = [&](const float* x, unsigned row, unsigned rows, unsigned ld, unsigned width) __attribute__((always_inline)) {
    const unsigned left = row < rows ? rows - row : 0;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x) + (size_t)row * ld, 0, left == 0 ? 0 : (int)(((left - 1) * ld + width) * 4u), 0x00020000);
  };
  auto four = [](__amdgpu_buffer_rsrc_t from, unsigned at) __attribute__((always_inline)) {
    return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0));
  };
  const bool masked = p.mask != nullptr;
  const float* const mask = masked ? p.mask + (size_t)bo * p.outerM + (size_t)bn * p.innerM : nullptr;
  unsigned ofK[GROUPS][QUADS], ofV[GROUPS][4];
#pragma unroll
  for (int b = 0; b < GROUPS; ++b)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ofK[b][j] = 16 * j + 4 * q < D ? ((16 * b + l16) * p.ldk + 16 * j + 4 * q) * 4u : kPastEnd;
      ofV[b][j] = 4 * l16 < D ? ((16 * b + 4 * q + j) * p.ldv + 4 * l16) * 4u : kPastEnd;
    }
  v4f qreg[BLOCKS][QUADS], kreg[GROUPS][QUADS], vreg[GROUPS][4];
  float mk[GROUPS][4] = {};
  auto load_k = [&](unsigned t0) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rk = rows_from(K, t0, T, p.ldk, D);
#pragma unroll
    for (int b = 0; b < GROUPS; ++b)
#pragma unroll
      for (int j = 0; j < QUADS; ++j) kreg[b][j] = four(rk, ofK[b][j]);
    if (masked) {
      const __amdgpu_buffer_rsrc_t rm = rows_from(mask, t0, T, 1, 1);
#pragma unroll
      for (int b = 0; b < GROUPS; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          mk[b][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rm, (16 * b + 4 * q + r) * 4u, 0, 0));
    }
  };
  auto load_v = [&](unsigned t0) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rv = rows_from(V, t0, T, p.ldv, D);
#pragma unroll
    for (int b = 0; b < GROUPS; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) vreg[b][r] = four(rv, ofV[b][r]);
  };
  const __amdgpu_buffer_rsrc_t rq = rows_from(Q, s0, S, p.ldq, D);
#pragma unroll
  for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
    for (int j = 0; j < QUADS; ++j)
      qreg[n][j] = four(rq, 16 * j + 4 * q < D ? ((16 * n + l16) * p.ldq + 16 * j + 4 * q) * 4u : kPastEnd);
  load_k(wave * RUN);
  load_v(wave * RUN);

  // a divisor that is a power of two divides exactly like a multiplication by its reciprocal
  const float divisor = p.divisor;
  const unsigned bits = __builtin_bit_cast(unsigned, divisor), expo = (bits >> 23) & 0xffu;
  const bool exact = (bits & 0x007fffffu) == 0 && expo >= 2 && expo <= 252;
  const bool dividing = p.divide && !exact;
  const float factor = p.divide && exact ? 1.0f / divisor : 1.0f;
  // over the four lanes that share a query
  auto over_groups = [](float v, auto join) __attribute__((always_inline)) {
    float a, b;
    butterfly_pair<32>(v, a, b); v = join(a, b);
    butterfly_pair<16>(v, a, b); return join(a, b);
  };
  float m[BLOCKS], l[BLOCKS];  // l: of this lane's keys
  v4f o[BLOCKS][4];
#pragma unroll
  for (int n = 0; n < BLOCKS; ++n) {
    m[n] = -FLT_MAX;
    l[n] = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[n][e] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  for (unsigned t0 = wave * RUN; t0 < T; t0 += WAVES * RUN) {
    v4f s[BLOCKS][GROUPS];
#pragma unroll
    for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
      for (int b = 0; b < GROUPS; ++b) s[n][b] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < QUADS; ++j) {
      if ((unsigned)(16 * j) >= D) break;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
          for (int b = 0; b < GROUPS; ++b) s[n][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kreg[b][j][e], qreg[n][j][e], s[n][b], 0, 0, 0);
    }
    float v[BLOCKS][GROUPS][4];
#pragma unroll
    for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
      for (int b = 0; b < GROUPS; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = s[n][b][r];
          v[n][b][r] = x * factor;
        }
    auto every = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
        for (int b = 0; b < GROUPS; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) v[n][b][r] = f(v[n][b][r], b, r);
    };
    if (dividing) every([&](float x, int, int) { return x / divisor; });
    if (masked) every([&](float x, int b, int r) { return x + mk[b][r]; });
    // what is no key weighs nothing, whatever the maximum
    if (t0 + RUN > T) every([&](float x, int b, int r) { return t0 + 16 * b + 4 * q + r < T ? x : -__builtin_inff(); });
    load_k(t0 + WAVES * RUN);
#pragma unroll
    for (int n = 0; n < BLOCKS; ++n) {
      float highest = m[n];
#pragma unroll
      for (int b = 0; b < GROUPS; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) highest = fmaxf(highest, v[n][b][r]);
      highest = over_groups(highest, [](float a, float b) { return fmaxf(a, b); });
      const float scale = softmax_exp(m[n] - highest);  // (in front of the first run there is nothing to scale)
      m[n] = highest;
      float sum = 0.f;
#pragma unroll
      for (int b = 0; b < GROUPS; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[n][b][r] = softmax_exp(v[n][b][r] - highest);
          sum += v[n][b][r];
        }
      l[n] = l[n] * scale + sum;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[n][e][r] *= scale;
    }
#pragma unroll
    for (int b = 0; b < GROUPS; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int n = 0; n < BLOCKS; ++n)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[n][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vreg[b][r][e], v[n][b][r], o[n][e], 0, 0, 0);
    load_v(t0 + WAVES * RUN);
  }

  // ---- the wavefronts meet
#pragma unroll
  for (int n = 0; n < BLOCKS; ++n) {
    l[n] = over_groups(l[n], [](float a, float b) { return a + b; });
    if (q == 0) {
      wm[wave][16 * n + l16] = m[n];
      wl[wave][16 * n + l16] = l[n];
    }
  }
  __syncthreads();
  float total[BLOCKS];
#pragma unroll
  for (int n = 0; n < BLOCKS; ++n) {
    float highest = -FLT_MAX;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) highest = fmaxf(highest, wm[w][16 * n + l16]);
    total[n] = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) total[n] += wl[w][16 * n + l16] * softmax_exp(wm[w][16 * n + l16] - highest);
    const float scale = softmax_exp(m[n] - highest);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v4f x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = o[n][e][r] * scale;
      part[wave][n][r][lane] = x;
    }
  }
  __syncthreads();
  const unsigned col = 16 * q + 4 * wave;
  if (col >= D) return;
#pragma unroll
  for (int n = 0; n < BLOCKS; ++n) {
    v4f sum = part[0][n][wave][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += part[w][n][wave][lane];
    sum *= 1.0f / total[n];  // one division per row, as in the stand-alone softmax
    const unsigned row = s0 + 16 * n + l16;
    if (row < S) __builtin_memcpy(O + (size_t)row * p.ldo + col, &sum, 16);
  }
}

const char* unsupported(const tfcc_rocm_attention_desc* d) {
  // a lone product of at most eight rows runs on the streaming kernel (sgemv.hip), whose sums are ordered differently
  if (d->s <= 8 && (unsigned long long)d->batch_outer * d->batch_inner == 1) return "a single head of at most eight query rows";
  if (d->d > (unsigned)kMaxD) return "head width above 64";
  if (d->d % 4 != 0) return "head width not a multiple of 4";
  if (d->ldq % 4 || d->ldk % 4 || d->ldv % 4) return "row stride not a multiple of 4 elements";
  if (d->stride_q % 4 || d->stride_k % 4 || d->stride_v % 4 || d->inner_stride_q % 4 || d->inner_stride_k % 4 ||
      d->inner_stride_v % 4)
    return "batch stride not a multiple of 4 elements";
  if ((uintptr_t)d->q % 16 || (uintptr_t)d->k % 16 || (uintptr_t)d->v % 16) return "operand not 16-byte aligned";
  const unsigned long long rows = d->s > d->t ? d->s : d->t, ld = d->ldq > d->ldk ? (d->ldq > d->ldv ? d->ldq : d->ldv)
                                                                                  : (d->ldk > d->ldv ? d->ldk : d->ldv);
  if (rows * ld + d->d >= (1ull << 28)) return "one batch entry spans 2^28 elements or more";
  return nullptr;
}

}  // namespace
}  // namespace tfcc_rocm

using namespace tfcc_rocm;

extern "C" int tfcc_rocm_attention_f32_supported(const tfcc_rocm_attention_desc* d) {
  return d != nullptr && unsupported(d) == nullptr ? 1 : 0;
}

extern "C" int tfcc_rocm_attention_f32(void* stream, const tfcc_rocm_attention_desc* d) {
  TFCC_REQUIRE(d != nullptr, "attention: null descriptor");
  TFCC_REQUIRE(d->q && d->k && d->v && d->out, "attention: null operand");
  TFCC_REQUIRE(d->s > 0 && d->t > 0 && d->d > 0 && d->batch_outer > 0 && d->batch_inner > 0, "attention: empty operand");
  TFCC_REQUIRE(d->ldq >= d->d && d->ldk >= d->d && d->ldv >= d->d && d->ldo >= d->d,
               "attention: row stride shorter than a row");
  const char* why = unsupported(d);
  TFCC_REQUIRE(why == nullptr, "attention: %s (use the separate products and softmax)", why);
  AttentionParams p{};
  p.Q = d->q; p.K = d->k; p.V = d->v; p.O = d->out;
  p.S = d->s; p.T = d->t; p.D = d->d;
  p.ldq = d->ldq; p.ldk = d->ldk; p.ldv = d->ldv; p.ldo = d->ldo;
  p.outerQ = d->stride_q; p.outerK = d->stride_k; p.outerV = d->stride_v; p.outerO = d->stride_out;
  p.innerQ = d->inner_stride_q; p.innerK = d->inner_stride_k; p.innerV = d->inner_stride_v; p.innerO = d->inner_stride_out;
  p.batchInner = d->batch_inner;
  int cus = 0;
  {
    int dev = 0;
    TFCC_HIP_CHECK(hipGetDevice(&dev));
    static int cuCount[16] = {};
    TFCC_REQUIRE(dev >= 0 && dev < 16, "device index %d", dev);
    if (!cuCount[dev]) TFCC_HIP_CHECK(hipDeviceGetAttribute(&cuCount[dev], hipDeviceAttributeMultiprocessorCount, dev));
    cus = cuCount[dev];
  }
  const attention_plan::Kernel kernel = attention_plan::kernel_of(d->s, d->t, (unsigned long long)d->batch_outer * d->batch_inner, cus);
  const unsigned rowsPerBlock = attention_plan::rows_of(kernel);
  p.blocksS = (d->s + rowsPerBlock - 1) / rowsPerBlock;
  const unsigned long long total = (unsigned long long)p.blocksS * d->batch_outer * d->batch_inner;
  TFCC_REQUIRE(total < (1ull << 31) - 8, "attention: too many blocks");
  p.total = (unsigned)total;
  p.chunk = (p.total + 7) / 8;
  const UDiv blocksDiv = udiv_prepare(p.blocksS), innerDiv = udiv_prepare(p.batchInner);
  p.blocksMagic = blocksDiv.magic; p.blocksShift = blocksDiv.shift;
  p.innerMagic = innerDiv.magic; p.innerShift = innerDiv.shift;
  p.divisor = d->divisor;
  p.divide = d->has_divisor ? 1 : 0;
  p.mask = d->mask;
  p.outerM = d->stride_mask;
  p.innerM = d->inner_stride_mask;
  constexpr size_t ldsBytes = (size_t)kLdsFloats * sizeof(float);
  static_assert(ldsBytes <= 80 * 1024, "two workgroups per CU");
  constexpr size_t ldsBytes32 = (size_t)(kMaxT * kPitchV + 32 * kPitchS) * sizeof(float);
  static_assert(3 * ldsBytes32 <= 160 * 1024, "three workgroups per CU");
  static bool attrSet[16] = {};
  int dev = 0;
  TFCC_HIP_CHECK(hipGetDevice(&dev));
  TFCC_REQUIRE(dev >= 0 && dev < 16, "device index %d", dev);
  if (!attrSet[dev]) {
    TFCC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(attention_kernel<64>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldsBytes));
    TFCC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(attention_kernel<32>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldsBytes32));
    attrSet[dev] = true;
  }
  const dim3 grid(p.chunk * 8), block(attention_plan::threads_of(kernel));
  switch (kernel) {
    case attention_plan::kRows64: hipLaunchKernelGGL(attention_kernel<64>, grid, block, ldsBytes, as_stream(stream), p); break;
    case attention_plan::kRows32: hipLaunchKernelGGL(attention_kernel<32>, grid, block, ldsBytes32, as_stream(stream), p); break;
    case attention_plan::kRows16:
      hipLaunchKernelGGL(d->t <= 64 ? attention_rows16_kernel<64> : attention_rows16_kernel<128>, grid, block, 0, as_stream(stream), p);
      break;
    case attention_plan::kRuns16: hipLaunchKernelGGL(attention_stream_kernel<1>, grid, block, 0, as_stream(stream), p); break;
    case attention_plan::kRuns32: hipLaunchKernelGGL(attention_stream_kernel<2>, grid, block, 0, as_stream(stream), p); break;
  }
  return check_launch("attention");
}
