// A whole LSTM sequence, or both directions of a bidirectional one, in one launch.
//
// The recurrence is a chain of small steps: [batch, units] times [units, 4 units], the cell, and every unit needs every
// unit's result of the step before.  A launch per step costs 4.8 us (4 x 512) although its arithmetic takes 0.2 us,
// because the state kernel is fetched again and the launch itself has to be paid.  Here a workgroup owns eight units for
// the whole sequence, keeps their columns of the state kernel in registers, and the workgroups hand their part of h to
// each other through memory: 2.1 us per step of 4 x 512, both directions at once (3.0 for 4 x 1024).  What is left is
// the way of h to memory and back and the polls that came too early.  Up to 768 units a second form keeps h inside an XCD:
// 1.4 us per step (lstm_xcd_kernel, below); the first one then takes what is recorded in a
// graph, and what a part of a partitioned GPU gets.
//
// The exchange is made of words that a reader polls themselves, so nothing is ordered by fences.  There are two kinds:
//   Up to 256 units, and in the second form, 64-bit words of a value and the number of the step it belongs to: a reader waits
//   for its step.  Two sets of words alternate; a workgroup writes step t + 2 only after it has read all of step t + 1, which every other
//   workgroup wrote after it had read all of step t, so no word is overwritten before its last reader is through.
//   With more units half the bytes, and a quarter of the loads, make up for one more store: 32-bit words, a value each,
//   four to a load.  One that has not been written holds kUnwritten.  Four sets take turns.  A workgroup that has read all
//   of step t knows that everyone has read all of step t - 1; behind its results for step t + 1 it clears its words of step
//   t - 1, has seen that clearing done before it stores its results for step t + 2, and those are what a reader has to have
//   before it looks at the cleared words again, for step t + 3.
// Served bidirectional sequences in the first form, us, all in 64-bit words before: 64 of 4 x 512 218 -> 213, 31 of 7 x 600
// 206 -> 183, 64 of 4 x 1024 327 -> 301, 32 of 12 x 1024 448 -> 345; in 32-bit words 64 of 1 x 256 take 141 against 131.
//
// All workgroups have to run at the same time.  The launcher asks for at most one per CU, but other work may hold CUs, so
// every wait is bounded: a workgroup that has waited `waitTicks` raises a flag and ends, the others see the flag and end,
// and the launch behind this one, which does nothing otherwise, finds the flag and computes the sequence in one workgroup
// per direction.
//
// Arithmetic: tfcc/core/operations/tfcc_rnn.cpp:29-135 with the cell of tfcc/mkl/kernel/tfcc_mklcellkernel.hpp:51-87.
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "lstm_sequence_plan.hpp"

namespace tfcc_rocm {
namespace {

struct Sequence {
  const float* x;       // [seq, batch, 4 units]: products of the inputs, gates i, c, f, o
  const float* kernel;  // [units, 4 units]
  const float* bias;    // [4 units]
  const float* h0;      // [batch, units]
  const float* c0;
  float* out;           // [seq, batch, units], in the order the steps are taken
  float* h;             // [batch, units]
  float* c;
  int backward;
};
struct SequenceParams {
  Sequence s[2];
  unsigned seq, batch, units, directions;
  float forget;
  unsigned blocksPerDirection;
  unsigned groups, rowsPerGroup;  // of the form with an XCD for a group of rows; none: the other one
  unsigned spread;                // that form with the workgroups of a group side by side, so on all XCDs
  unsigned* words;  // [set][direction][batch][pitch]
  unsigned* failed;
  unsigned long long waitTicks;
  int naps;  // before the first poll of a step
};

__device__ __forceinline__ float sigmoid_value(float v) { return 1.f / (1.f + expf(0.f - v)); }

constexpr unsigned kUnwritten = 0xffffffffu;  // (a NaN; another one goes in its place where a value is just this)
__device__ __forceinline__ unsigned word_of(float value) {
  const unsigned bits = __builtin_bit_cast(unsigned, value);
  return bits == kUnwritten ? 0x7fc00000u : bits;
}

__device__ __forceinline__ unsigned long long numbered_word(float value, unsigned step) {
  return ((unsigned long long)step << 32) | __builtin_bit_cast(unsigned, value);
}
constexpr unsigned kStepMask = 0x0fffffffu;  // where the words of a step carry the XCD they come from above it
using lstm_plan::kXcds;
constexpr bool numbered(unsigned pitch) { return pitch <= 256; }  // 64-bit words, with the number of the step

// Step 0 reads the initial h from the first set (as words of step 1); the others hold nothing anybody waits for.  Units that
// do not exist are zeros in every set.
__global__ __launch_bounds__(256) void lstm_exchange_init_kernel(SequenceParams p, unsigned pitch, unsigned total, bool withNumbers) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i == 0) *p.failed = 0;
  if (i >= total) return;
  const unsigned u = i % pitch, b = i / pitch % p.batch, d = i / pitch / p.batch;
  const float h = u < p.units ? p.s[d].h0[(size_t)b * p.units + u] : 0.f;
  if (withNumbers) {
    reinterpret_cast<unsigned long long*>(p.words)[i] = numbered_word(h, 1);
    reinterpret_cast<unsigned long long*>(p.words)[(size_t)total + i] = 0;
    return;
  }
  p.words[i] = word_of(h);
  for (unsigned set = 1; set < 4; ++set) p.words[(size_t)set * total + i] = u < p.units ? kUnwritten : 0u;
}

// Sums v[0 .. N) over the lanes that differ in the bits MASK, MASK / 2, ..., U of their number.  While the count is
// even, the two halves of a pair of lanes keep one half of the values each: a lane ends with the totals of the values
// base .. base + left(N) - 1.
template <int N, int MASK, int U>
constexpr int values_left() {
  if constexpr (MASK >= U) return values_left<(N % 2 == 0 ? N / 2 : N), MASK / 2, U>();
  else return N;
}
template <int N, int MASK, int U, int TOTAL>
__device__ __forceinline__ void sum_over_lanes(float (&v)[TOTAL], int lane, int& base) {
  if constexpr (MASK >= U) {
    if constexpr (N % 2 == 0) {
      constexpr int HALF = N / 2;
      const bool upper = (lane & MASK) != 0;
#pragma unroll
      for (int a = 0; a < HALF; ++a) {
        if constexpr (MASK >= 16) {
          const unsigned x = __builtin_bit_cast(unsigned, v[a]), y = __builtin_bit_cast(unsigned, v[a + HALF]);
          unsigned r0, r1;
          if constexpr (MASK == 32) {
            const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
            r0 = (unsigned)r[0]; r1 = (unsigned)r[1];
          } else {
            const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
            r0 = (unsigned)r[0]; r1 = (unsigned)r[1];
          }
          v[a] = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
        } else {
          const float mine = upper ? v[a + HALF] : v[a], theirs = upper ? v[a] : v[a + HALF];
          float same, other;
          butterfly_pair<MASK>(theirs, same, other);
          v[a] = mine + other;
        }
      }
      base += upper ? HALF : 0;
      sum_over_lanes<HALF, MASK / 2, U>(v, lane, base);
    } else {
#pragma unroll
      for (int a = 0; a < N; ++a) {
        float x, y;
        butterfly_pair<MASK>(v[a], x, y);
        v[a] = x + y;
      }
      sum_over_lanes<N, MASK / 2, U>(v, lane, base);
    }
  }
}

// the value that lane LANE of this lane's quad holds (through LDS, as a shuffle: 20 ns more per step)
template <int LANE>
__device__ __forceinline__ float of_quad(float v) {
  const int x = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(x, x, LANE * 0x55, 0xf, 0xf, false));
}

typedef float lstm_v4f __attribute__((ext_vector_type(4)));
typedef unsigned lstm_v4u __attribute__((ext_vector_type(4)));

constexpr unsigned kNothing = 0x80000000u;  // an offset past every set: reads zeros without a trip to memory
constexpr int kDeviceScope = 16;            // sc1, as a load of an atomic at device scope has it

// The cell's functions stand in the chain of every step, so they are written without branches and share an exponential and
// a quotient: with e = e^-|v|, sigmoid(v) = 1 / (1 + e), or e / (1 + e) for negative v, and with e = e^-2|v|, tanh(v) =
// (1 - e) / (1 + e) with v's sign.  What the sum and the difference round off (exactly known, as e <= 1) goes into the one
// correction of the quotient, so that little but the error of e is left.  Below 0.65, where the difference would bring that
// out, tanh is v + v^3 P(v^2), with P of degree 5 fitted for the smallest relative error (tests/golden/fit_tanh.py makes
// the coefficients).  The exponential of x <= 0: x log2(e) = n + t with a whole n and |t| <= 1/2, t with what the constant
// leaves out added, then 2^t by the hardware, times 2^n; 0 below -104, NaN stays NaN.
//
// Closer to the exact values than the library's expf and tanhf in the plain formulas; largest / mean error in units in the
// last place: tanh on 0.5 .. 0.7 0.9 / 0.26 against 1.4 / 0.30, on 1 .. 10 0.8 / 0.24 against 1.3 / 0.24, sigmoid on -4 .. 4
// 1.6 / 0.29 against 2.1 / 0.41, on -20 .. -4 1.4 / 0.34 against 2.4 / 0.38.
__device__ __forceinline__ float sigmoid_or_tanh(float v, bool tanhWanted) {
  const float y = __builtin_fabsf(v);
  float x = tanhWanted ? -2.f * y : -y;
  x = x < -104.f ? -104.f : x;
  const float L = 1.44269504088896341f;
  const float n = __builtin_rintf(x * L);
  const float part = __builtin_amdgcn_exp2f(fmaf(x, 1.92596303e-8f, fmaf(x, L, -n))), scale = __builtin_ldexpf(1.f, (int)n);
  const float den = fmaf(part, scale, 1.f), r = __builtin_amdgcn_rcpf(den);
  const float e = part * scale, denRest = e - (den - 1.f), diff = 1.f - e;
  const float num = tanhWanted ? diff : v < 0.f ? e : 1.f, numRest = tanhWanted ? (1.f - diff) - e : 0.f;
  float q = num * r;
  q = fmaf(fmaf(-den, q, num) + fmaf(-denRest, q, numRest), r, q);
  const float s = v * v;
  float p = 2.059580758e-03f;
  p = fmaf(p, s, -8.085626177e-03f);
  p = fmaf(p, s, 2.166340314e-02f);
  p = fmaf(p, s, -5.393994227e-02f);
  p = fmaf(p, s, 1.333315223e-01f);
  p = fmaf(p, s, -3.333332837e-01f);
  const float small = fmaf(v * s, p, v);
  return tanhWanted && y < 0.65f ? small : __builtin_copysignf(q, tanhWanted ? v : 1.f);
}

// A wavefront owns a unit and sums its four gates over all of K = 64 KI rows of the state kernel for 4 Q rows of the
// batch, with matrix ops of sixteen independent 4 x 4 x 1 blocks: block = lane / 4 takes the rows k = 64 i + 4 block + r,
// the four columns are the gates, the four rows four rows of the batch.  Twice the rate of the vector unit, no rows or
// columns of padding at four rows, and what remains, sixteen partial sums of 4 Q values, ends one value per lane with the
// four gates of a unit side by side: the wavefront finishes its unit alone, and the only barrier of a step is the one
// behind the exchange (on the vector unit, with the sums joined through LDS: 3.0 us per step against 2.3).
template <int Q, int KI, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void lstm_sequence_kernel(SequenceParams p) {
  constexpr int T = 64 * WAVES, K = 64 * KI, MB = 4 * Q, LP = K + 16;  // LP: four rows fall on different banks
  constexpr int LEFT = values_left<MB, 32, 4>();
  extern __shared__ __attribute__((aligned(16))) float hs[];  // [2][MB][LP]
  __shared__ int gaveUp;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned units = p.units, batch = p.batch;
  const unsigned d = blockIdx.x / p.blocksPerDirection;
  const Sequence& s = p.s[d];
  constexpr bool NUMBERED = numbered(K);
  constexpr unsigned SIZE = NUMBERED ? 2 : 1;  // of a word, in 32 bits
  const size_t setSize = (size_t)p.directions * batch * K * SIZE;
  unsigned* const mine = p.words + (size_t)d * batch * K * SIZE;
  for (int i = tid; i < 2 * MB * LP; i += T) hs[i] = 0.f;  // rows of the batch and units that do not exist stay zero
  if (tid == 0) gaveUp = p.waitTicks == 0;  // no wait at all: the launch behind this one has the sequence
  __syncthreads();

  const unsigned u = (blockIdx.x - d * p.blocksPerDirection) * WAVES + wave;
  const int gate = lane & 3, block = lane >> 2;
  const bool exists = u < units;
  float w[KI][4];
#pragma unroll
  for (int i = 0; i < KI; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned k = 64 * i + 4 * block + r;
      w[i][r] = (k < units && exists) ? s.kernel[(size_t)k * 4 * units + (size_t)gate * units + u] : 0.f;
    }
  // the row of the batch whose values this lane finishes
  int base = 0;
  {
    float none[MB] = {};
    sum_over_lanes<MB, 32, 4>(none, lane, base);
  }
  // what the halving has not told apart are copies: the first LEFT of the lanes that hold the same values take one each
  constexpr int COPIES = 16 / (MB / LEFT);  // lanes of a gate that hold the same LEFT values
  const int copy = block & (COPIES - 1);
  const unsigned fm = base + (LEFT > 1 ? copy : 0);
  const bool valid = copy < LEFT && fm < batch && exists;
  auto inputOf = [&](unsigned step) {
    const unsigned t = s.backward ? p.seq - 1 - step : step;
    return valid ? s.x[((size_t)t * batch + fm) * 4 * units + (size_t)gate * units + u] : 0.f;
  };
  const size_t at = (size_t)fm * units + u;
  const float bv = valid ? s.bias[(size_t)gate * units + u] : 0.f;
  float cPrev = valid ? s.c0[at] : 0.f, xin = inputOf(0);
  const float forget = gate == 2 ? p.forget : -0.f;  // (adding -0 changes nothing)

  for (unsigned step = 0; step < p.seq; ++step) {
    // ---- h of the step before: every thread polls its words.  (Two buffers in LDS: a slow wavefront may still read the
    // last step's.)  A poll that comes too early costs a whole trip to memory before the next one, and the traffic holds
    // up the words it waits for; that the polling wavefronts are the ones that have just finished a step is what keeps
    // most first polls from coming too early (wavefronts that only poll: 4.9 us per step against 2.3).
    float* h = hs + (step & 1u) * (MB * LP);
    if constexpr (NUMBERED) {
      const unsigned long long* words = reinterpret_cast<const unsigned long long*>(mine) + (step & 1u) * (setSize / 2);
      if constexpr (Q > 2) __builtin_amdgcn_s_sleep(2);
      const unsigned long long start = wall_clock64();
      constexpr int PER = (MB * K + T - 1) / T;
      unsigned long long v[PER];
      bool wanted[PER];
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const unsigned i = tid + k * T;
        wanted[k] = i < batch * K && i % K < units;
      }
      for (unsigned tries = 0;; ++tries) {
        bool ready = true;
#pragma unroll
        for (int k = 0; k < PER; ++k)
          v[k] = wanted[k] ? __hip_atomic_load(words + tid + k * T, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
#pragma unroll
        for (int k = 0; k < PER; ++k) ready = ready && (!wanted[k] || (unsigned)(v[k] >> 32) == step + 1);
        if (ready) break;
        if ((tries & 15u) == 15u &&
            (wall_clock64() - start > p.waitTicks ||
             __hip_atomic_load(p.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          gaveUp = 1;
          break;
        }
      }
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const unsigned i = tid + k * T;
        if (wanted[k]) h[i / K * LP + i % K] = __builtin_bit_cast(float, (unsigned)v[k]);
      }
    } else {
      const unsigned* set = mine + (step & 3u) * setSize;
      for (int i = 0; i < p.naps; ++i) __builtin_amdgcn_s_sleep(2);
      const unsigned long long start = wall_clock64();
      const __amdgpu_buffer_rsrc_t words = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned*>(set), 0, (int)(batch * K * 4), 0x00020000);
      constexpr int PER = (MB * K / 4 + T - 1) / T;
      unsigned wanted[PER];  // byte offsets; kNothing: there, or never wanted
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const unsigned i = 4 * (tid + k * T);
        wanted[k] = i < batch * K && i % K < units ? i * 4u : kNothing;
      }
      for (unsigned tries = 0;; ++tries) {
        asm volatile("" ::: "memory");  // every try asks memory again
        lstm_v4u v[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k)
          v[k] = __builtin_bit_cast(lstm_v4u, __builtin_amdgcn_raw_buffer_load_b128(words, wanted[k], 0, kDeviceScope));
        bool ready = true;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
          const unsigned i = 4 * (tid + k * T);
          const bool written = v[k][0] != kUnwritten && v[k][1] != kUnwritten && v[k][2] != kUnwritten && v[k][3] != kUnwritten;
          if (wanted[k] != kNothing && written) {
            *reinterpret_cast<lstm_v4u*>(h + i / K * LP + i % K) = v[k];
            wanted[k] = kNothing;
          }
          ready = ready && wanted[k] == kNothing;
        }
        if (ready) break;
        if ((tries & 15u) == 15u &&
            (wall_clock64() - start > p.waitTicks ||
             __hip_atomic_load(p.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          gaveUp = 1;
          break;
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's stores of the step before are done
    }
    __syncthreads();
    if (gaveUp) {  // the same for the whole workgroup
      if (tid == 0) __hip_atomic_store(p.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }

    // ---- the wavefront's four columns of h times the state kernel; the next step's inputs are asked for now, because
    // the words polled next can only return behind them
    const bool last = step + 1 == p.seq;
    const float xNext = last ? 0.f : inputOf(step + 1);
    constexpr int CHAINS = Q == 1 ? 2 : 1;  // accumulators per sum: a matrix op waits for the one before it on its own
    lstm_v4f acc[Q][CHAINS];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int c = 0; c < CHAINS; ++c) acc[q][c] = lstm_v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < KI; ++i)
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const lstm_v4f a = *reinterpret_cast<const lstm_v4f*>(h + (4 * q + gate) * LP + 64 * i + 4 * block);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[q][r % CHAINS] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[r], w[i][r], acc[q][r % CHAINS], 0, 0, 0);
      }
    float v[MB];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[4 * q + r] = acc[q][0][r];
#pragma unroll
        for (int c = 1; c < CHAINS; ++c) v[4 * q + r] += acc[q][c][r];
      }
    int unused = 0;
    sum_over_lanes<MB, 32, 4>(v, lane, unused);
    float sum = v[0];
#pragma unroll
    for (int a = 1; a < LEFT; ++a) sum = copy == a ? v[a] : sum;

    // ---- the cell
    const float pre = xin + sum + bv + forget;
    const float act = sigmoid_or_tanh(pre, gate == 1);
    // the four gates of a unit lie in one quad of lanes
    const float xi = of_quad<0>(act), xc = of_quad<1>(act), xf = of_quad<2>(act), xo = of_quad<3>(act);
    const float c = __fadd_rn(__fmul_rn(xc, xi), __fmul_rn(cPrev, xf)), hn = sigmoid_or_tanh(c, true) * xo;
    cPrev = c;
    xin = xNext;
    if (valid && gate == 0) {
      if constexpr (NUMBERED) {
        if (!last)
          __hip_atomic_store(reinterpret_cast<unsigned long long*>(mine) + ((step + 1) & 1u) * (setSize / 2) + (size_t)fm * K + u,
                             numbered_word(hn, step + 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        unsigned* const word = mine + (size_t)fm * K + u;
        if (!last) __hip_atomic_store(word + ((step + 1) & 3u) * setSize, word_of(hn), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (step > 0) __hip_atomic_store(word + ((step - 1) & 3u) * setSize, kUnwritten, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      s.out[(size_t)step * batch * units + at] = hn;
      if (last) {
        s.h[at] = hn;
        s.c[at] = c;
      }
    }
  }
}

// The XCD that a wavefront runs on: four bits of the register XCC_ID.
__device__ __forceinline__ unsigned xcd_id() { return __builtin_amdgcn_s_getreg(20 | (3 << 11)); }

// The form for up to 768 units on a whole GPU: the state kernel of a direction fits the registers of one XCD's 32 CUs, 16, 64
// or 144 of a lane, so nothing has to leave the XCD between two steps, and the rows of the batch, which do not need one
// another, are dealt out to the XCDs, four groups of them to each of two directions, eight to one.  A store that stops in the XCD's L2
// and a load at device scope, which looks there first, take 0.78 us from all to all of 32 workgroups with 32 words each,
// where a store to memory takes 1.16, and 1.38 with the workgroups on eight XCDs.
//
// That the workgroups of a group share an XCD is what the dispatch of workgroups to XCDs in turn gives; nothing depends on
// it but time.  The words of the first step go through to memory and carry the XCD they come from; everyone reads all of them,
// so everyone knows whether they are all from one, and if not, h goes through to memory in all steps.
//
// In the terms of the memory model a store for the workgroup hands nothing to another workgroup, whatever XCD it runs on.  That it is
// seen rests on this chip: such a store goes to the L2, which is where a load at device scope looks.  What does not rest on it
// is the result: a word is taken only with its step's number, which its value came with in one store of 64 bits, so what is not
// seen, or seen late, can only end a wait, and then the launch behind computes the sequence.
//
// A wavefront owns UPW units.  A lane takes four k in 256 of all their gates, so a row of h is KQ loads from LDS, and
// the products are on the vector unit: one row leaves three of the four rows of a 4 x 4 x 1 matrix op empty, and with four the
// time is the same.  100 steps of both directions, us, the form above -> this one: 1 x 128 162 -> 119, 4 x 256 171 -> 122, 16 x 256
// 495 -> 158, 4 x 512 212 -> 139, 8 x 512 277 -> 182, 16 x 512 484 -> 243, 4 x 768 265 -> 192, 12 x 700 446 -> 332; one step of 4 x
// 512 19.5 -> 11.5.  Of 1.5 us for a step of 4 x 512 the products take 0.26 when they are left out, the cell's functions 0.28, inputs and results 0.15;
// the exchange and the rest is 0.88.  (The form above on one XCD, all rows in each: 4 x 512 2.0 a step, 8 x 512 2.7, 4 x 768 3.35.
// Words that have arrived not asked for again: 16 x 512 2.85 against 2.6.  Results stored a step later, or inputs fetched one
// step at a time, not four: 2.6 against 2.55.)
template <int ROWS, int KQ>
__global__ __launch_bounds__(512) void lstm_xcd_kernel(SequenceParams p) {
  constexpr int WAVES = 8, T = 64 * WAVES, K = 256 * KQ, UPW = KQ, SUMS = UPW * ROWS;
  constexpr int LEFT = values_left<SUMS, 32, 4>(), COPIES = 16 / (SUMS / LEFT);
  static_assert(LEFT <= COPIES, "a lane finishes one value");
  __shared__ __attribute__((aligned(16))) float hs[2][ROWS][K], columns[WAVES * UPW][260];  // (260: a wavefront's writes on all banks)
  __shared__ int gaveUp, apart;
  const unsigned members = gridDim.x / kXcds, turn = p.spread ? blockIdx.x / members : blockIdx.x % kXcds;
  const unsigned member = p.spread ? blockIdx.x - turn * members : blockIdx.x / kXcds, d = turn / p.groups, group = turn - d * p.groups;
  if (d >= p.directions) return;  // nothing for this XCD
  const int tid = threadIdx.x, lane = tid & 63, gate = lane & 3;
  const unsigned xcd = xcd_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned units = p.units, row0 = group * p.rowsPerGroup, rows = min(p.rowsPerGroup, p.batch - row0);
  const Sequence& s = p.s[d];
  const size_t setSize = (size_t)p.directions * p.batch * K;
  unsigned long long* const mine = reinterpret_cast<unsigned long long*>(p.words) + ((size_t)d * p.batch + row0) * K;
  for (int i = tid; i < 2 * ROWS * K; i += T) (&hs[0][0][0])[i] = 0.f;  // rows and units that do not exist stay zero
  if (tid == 0) {
    gaveUp = p.waitTicks == 0;  // no wait at all: the launch behind this one has the sequence
    apart = 0;
  }
  __syncthreads();

  const unsigned u0 = (member * WAVES + wave) * UPW;
  // The state kernel: rows of a gate's units side by side go through LDS, four values to a load (fetched by the lanes that keep
  // them, a value of a row at a time, 4 x 512 takes 12 us longer and 4 x 768 31).  Rows that do not exist are zeros; what
  // stands in the place of units that do not is nobody's.
  float w[KQ][4][4][UPW];  // [.][k][gate][unit]
  {
    const __amdgpu_buffer_rsrc_t kernel = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(s.kernel), 0, (int)(16u * units * units), 0x00020000);
    const unsigned first = member * (WAVES * UPW);
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
      lstm_v4f rows[4][UPW];
      auto place = [&](int n, unsigned& k, unsigned& unit) {  // 2 UPW loads side by side are a row
        const unsigned item = tid + n * T;
        k = item / (2 * UPW);
        unit = item % (2 * UPW) * 4;
      };
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int n = 0; n < UPW; ++n) {
          unsigned k, unit;
          place(n, k, unit);
          const unsigned at = ((256 * i + k) * 4 + g) * units + first + unit, end = 4 * units * units;
          rows[g][n] = __builtin_bit_cast(lstm_v4f, __builtin_amdgcn_raw_buffer_load_b128(kernel, 256 * i + k < units ? at * 4u : kNothing, 0, 0));
          if (at < end && at + 4 > end)  // the last row of the last gate: four values that the matrix ends in are not fetched at all
#pragma unroll
            for (unsigned e = 0; e < 3; ++e) rows[g][n][e] = at + e < end ? s.kernel[at + e] : 0.f;
        }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        __syncthreads();
#pragma unroll
        for (int n = 0; n < UPW; ++n) {
          unsigned k, unit;
          place(n, k, unit);
#pragma unroll
          for (int e = 0; e < 4; ++e) columns[unit + e][k] = rows[g][n][e];
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < UPW; ++n) {
          const lstm_v4f v = *reinterpret_cast<const lstm_v4f*>(&columns[wave * UPW + n][4 * lane]);
#pragma unroll
          for (int e = 0; e < 4; ++e) w[i][e][g][n] = v[e];
        }
      }
    }
  }
  // the unit and the row whose sum this lane ends with, as in the other form
  int base = 0;
  {
    float none[SUMS] = {};
    sum_over_lanes<SUMS, 32, 4>(none, lane, base);
  }
  const int copy = (lane >> 2) & (COPIES - 1);
  const unsigned finished = base + (LEFT > 1 ? copy : 0);  // [unit][row]
  const unsigned u = u0 + finished / ROWS, r = finished % ROWS, fm = row0 + r;
  const bool valid = copy < LEFT && r < rows && u < units;
  auto inputOf = [&](unsigned step) {
    const unsigned t = s.backward ? p.seq - 1 - step : step;
    return valid ? s.x[((size_t)t * p.batch + fm) * 4 * units + (size_t)gate * units + u] : 0.f;
  };
  const size_t at = (size_t)fm * units + u;
  const float bv = valid ? s.bias[(size_t)gate * units + u] : 0.f;
  float cPrev = valid ? s.c0[at] : 0.f;
  const float forget = gate == 2 ? p.forget : -0.f;  // (adding -0 changes nothing)
  constexpr int AHEAD = 4;
  float xin[AHEAD], xNext[AHEAD];
#pragma unroll
  for (int q = 0; q < AHEAD; ++q) xin[q] = (unsigned)q < p.seq ? inputOf(q) : 0.f;

  // false: someone has waited too long
  auto take = [&](unsigned step, auto q) __attribute__((always_inline)) -> bool {
    float (*h)[K] = hs[step & 1u];
    const unsigned long long* words = mine + (step & 1u) * setSize;
    const unsigned long long start = wall_clock64();
    constexpr int PER = (ROWS * K + T - 1) / T;
    unsigned long long v[PER];
    bool wanted[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const unsigned i = tid + k * T;
      wanted[k] = i < rows * K && i % K < units;
    }
    for (unsigned tries = 0;; ++tries) {
      bool ready = true;
#pragma unroll
      for (int k = 0; k < PER; ++k)
        v[k] = wanted[k] ? __hip_atomic_load(words + tid + k * T, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
#pragma unroll
      for (int k = 0; k < PER; ++k) ready = ready && (!wanted[k] || ((unsigned)(v[k] >> 32) & kStepMask) == step + 1);
      if (ready) break;
      if ((tries & 15u) == 15u &&
          (wall_clock64() - start > p.waitTicks ||
           __hip_atomic_load(p.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
        gaveUp = 1;
        break;
      }
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const unsigned i = tid + k * T;
      if (wanted[k]) h[i / K][i % K] = __builtin_bit_cast(float, (unsigned)v[k]);
      if (step == 1 && wanted[k] && (unsigned)(v[k] >> 60) != xcd) apart = 1;
    }
    __syncthreads();
    if (gaveUp) {  // the same for the whole workgroup
      if (tid == 0) __hip_atomic_store(p.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    const bool last = step + 1 == p.seq;
    if (q == 0) {
#pragma unroll
      for (unsigned n = 0; n < AHEAD; ++n) xNext[n] = step + AHEAD + n < p.seq ? inputOf(step + AHEAD + n) : 0.f;
    }

    float sum[4][SUMS];
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int n = 0; n < SUMS; ++n) sum[g][n] = 0.f;
#pragma unroll
    for (int i = 0; i < KQ; ++i)
#pragma unroll
      for (int b = 0; b < ROWS; ++b) {
        const lstm_v4f a = *reinterpret_cast<const lstm_v4f*>(&h[b][256 * i + 4 * lane]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int n = 0; n < UPW; ++n) sum[g][ROWS * n + b] = fmaf(a[e], w[i][e][g][n], sum[g][ROWS * n + b]);
      }
    // the four gates to the four lanes of a quad
    float half[2][SUMS], v1[SUMS];
    const bool odd = (lane & 1) != 0, upper = (lane & 2) != 0;
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int n = 0; n < SUMS; ++n) {
        float same, other;
        butterfly_pair<2>(upper ? sum[g][n] : sum[g + 2][n], same, other);
        half[g][n] = (upper ? sum[g + 2][n] : sum[g][n]) + other;
      }
#pragma unroll
    for (int n = 0; n < SUMS; ++n) {
      float same, other;
      butterfly_pair<1>(odd ? half[0][n] : half[1][n], same, other);
      v1[n] = (odd ? half[1][n] : half[0][n]) + other;
    }
    int unused = 0;
    sum_over_lanes<SUMS, 32, 4>(v1, lane, unused);
    float total = v1[0];
#pragma unroll
    for (int a = 1; a < LEFT; ++a) total = copy == a ? v1[a] : total;

    // ---- the cell
    const float act = sigmoid_or_tanh(xin[q] + total + bv + forget, gate == 1);
    const float xi = of_quad<0>(act), xc = of_quad<1>(act), xf = of_quad<2>(act), xo = of_quad<3>(act);
    const float c = __fadd_rn(__fmul_rn(xc, xi), __fmul_rn(cPrev, xf)), hn = sigmoid_or_tanh(c, true) * xo;
    cPrev = c;
    if (valid && gate == 0) {
      unsigned long long* const word = mine + ((step + 1) & 1u) * setSize + (size_t)r * K + u;
      if (!last) {
        const unsigned long long v = numbered_word(hn, step + 2) | (step == 0 ? (unsigned long long)xcd << 60 : 0ull);
        if (step == 0 || apart) __hip_atomic_store(word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else __hip_atomic_store(word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      s.out[(size_t)step * p.batch * units + at] = hn;
      if (last) {
        s.h[at] = hn;
        s.c[at] = c;
      }
    }
    return true;
  };
  for (unsigned step = 0; step < p.seq; step += AHEAD) {
    if (!take(step, std::integral_constant<int, 0>{})) return;
    if (step + 1 >= p.seq || !take(step + 1, std::integral_constant<int, 1>{})) return;
    if (step + 2 >= p.seq || !take(step + 2, std::integral_constant<int, 2>{})) return;
    if (step + 3 >= p.seq || !take(step + 3, std::integral_constant<int, 3>{})) return;
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) xin[n] = xNext[n];
  }
}

// The sequence once more in one workgroup per direction, if the launch before it gave up.
__global__ __launch_bounds__(1024) void lstm_repair_kernel(SequenceParams p) {
  if (__hip_atomic_load(p.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) return;
  const Sequence& s = p.s[blockIdx.x];
  const unsigned units = p.units, batch = p.batch, state = batch * units;
  for (unsigned i = threadIdx.x; i < state; i += 1024) s.c[i] = s.c0[i];
  for (unsigned step = 0; step < p.seq; ++step) {
    const float* h = step == 0 ? s.h0 : s.out + (size_t)(step - 1) * state;
    const unsigned t = s.backward ? p.seq - 1 - step : step;
    for (unsigned i = threadIdx.x; i < state; i += 1024) {
      const unsigned b = i / units, u = i - b * units;
      float sum[4] = {0.f, 0.f, 0.f, 0.f};
      for (unsigned r = 0; r < units; ++r)
        for (int q = 0; q < 4; ++q) sum[q] = fmaf(h[(size_t)b * units + r], s.kernel[(size_t)r * 4 * units + q * units + u], sum[q]);
      const float* x = s.x + ((size_t)t * batch + b) * 4 * units + u;
      float pre[4];
      for (int q = 0; q < 4; ++q) pre[q] = x[(size_t)q * units] + sum[q] + s.bias[(size_t)q * units + u];
      const float xi = sigmoid_value(pre[0]), xc = tanhf(pre[1]), xf = sigmoid_value(pre[2] + p.forget), xo = sigmoid_value(pre[3]);
      const float c = __fadd_rn(__fmul_rn(xc, xi), __fmul_rn(s.c[i], xf)), hn = tanhf(c) * xo;
      s.c[i] = c;
      s.out[(size_t)step * state + i] = hn;
      if (step + 1 == p.seq) s.h[i] = hn;
    }
    __threadfence_block();
    __syncthreads();
  }
}

template <int Q, int KI, int WAVES>
int launch(hipStream_t stream, SequenceParams p) {
  constexpr unsigned pitch = 64 * KI;
  static_assert(WAVES == (int)lstm_plan::kUnitsPerWorkgroup, "a wavefront per unit");
  constexpr size_t lds = (size_t)2 * 4 * Q * (pitch + 16) * sizeof(float);
  static_assert(lds <= 140 * 1024, "LDS budget");
  p.blocksPerDirection = lstm_plan::workgroups(p.units, 1);
  // The more words there are, the longer a poll takes, and one that comes too early holds up the words it waits for.  Us
  // with 0, 1, 4, 9 and 12 naps of 128 cycles: 32 steps of 12 x 1024 436, 429, 410, 344, 345; 40 of 8 x 1000 391, 373, 292,
  // 298, 302; 40 of 12 x 512 294, 286, 256, 256, 261; 40 of 5 x 600 211, 201, 204, 211, 218; 64 of 4 x 512 215, 217, 223, 238.
  const unsigned words = p.batch * pitch;
  p.naps = words <= 2048 ? 0 : words <= 4096 ? 1 : words <= 8192 ? 4 : 9;
  int dev = 0;
  TFCC_HIP_CHECK(hipGetDevice(&dev));
  TFCC_REQUIRE(dev >= 0 && dev < 16, "device index %d", dev);
  auto kern = lstm_sequence_kernel<Q, KI, WAVES>;
  static bool attrSet[16] = {};  // per device: the attribute belongs to the function on one device
  if (!attrSet[dev]) {
    TFCC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attrSet[dev] = true;
  }
  const unsigned total = p.directions * p.batch * pitch;
  hipLaunchKernelGGL(lstm_exchange_init_kernel, dim3((total + 255) / 256), dim3(256), 0, stream, p, pitch, total, numbered(pitch));
  hipLaunchKernelGGL(kern, dim3(p.blocksPerDirection * p.directions), dim3(64 * WAVES), lds, stream, p);
  hipLaunchKernelGGL(lstm_repair_kernel, dim3(p.directions), dim3(1024), 0, stream, p);
  return check_launch("lstm_sequence");
}

template <int ROWS, int KQ>
int launch_xcd(hipStream_t stream, const SequenceParams& p) {
  constexpr unsigned pitch = 256 * KQ;
  const unsigned total = p.directions * p.batch * pitch, workgroups = (p.units + 8 * KQ - 1) / (8 * KQ);
  hipLaunchKernelGGL(lstm_exchange_init_kernel, dim3((total + 255) / 256), dim3(256), 0, stream, p, pitch, total, true);
  hipLaunchKernelGGL((lstm_xcd_kernel<ROWS, KQ>), dim3(kXcds * workgroups), dim3(512), 0, stream, p);
  hipLaunchKernelGGL(lstm_repair_kernel, dim3(p.directions), dim3(1024), 0, stream, p);
  return check_launch("lstm_sequence");
}
template <int KQ>
int launch_xcd_rows(hipStream_t stream, const SequenceParams& p) {
  if (p.rowsPerGroup == 1) return launch_xcd<1, KQ>(stream, p);
  if (p.rowsPerGroup == 2) return launch_xcd<2, KQ>(stream, p);
  if (p.rowsPerGroup == 3) return launch_xcd<3, KQ>(stream, p);
  return launch_xcd<4, KQ>(stream, p);
}

template <int KI, int WAVES>
int launch_rows(hipStream_t stream, const SequenceParams& p) {
  if (p.batch <= 4) return launch<1, KI, WAVES>(stream, p);
  if (p.batch <= 8) return launch<2, KI, WAVES>(stream, p);
  if (p.batch <= 12) return launch<3, KI, WAVES>(stream, p);
  return launch<4, KI, WAVES>(stream, p);
}

int launch_units(hipStream_t stream, const SequenceParams& p) {
  if (p.rowsPerGroup != 0) {
    if (p.units <= 256) return launch_xcd_rows<1>(stream, p);
    if (p.units <= 512) return launch_xcd_rows<2>(stream, p);
    return launch_xcd_rows<3>(stream, p);
  }
  // eight wavefronts, so eight units, per workgroup: with four, twice the workgroups poll; with twelve or sixteen, each of
  // which reads all of h from LDS, that takes longer than the trip to memory (4 x 1024: 3.8, 5.8 and 7.0 us per step with
  // eight, twelve and sixteen)
  if (p.units <= 256) return launch_rows<4, 8>(stream, p);
  if (p.units <= 512) return launch_rows<8, 8>(stream, p);
  return launch_rows<16, 8>(stream, p);
}

// Two of these launches at once would each hold CUs that the other waits for, until both give up: launches from different
// streams of the process follow one another.  Once a second stream has turned up, each leaves an event on the stream that
// ran it for the next one to wait for, so no stream is looked at that may be gone, or is being captured, by then.  (Before
// that nothing is recorded, which a short sequence would feel: 2.7 us of 33 for 4 steps of 2 x 64.  The second stream's
// first sequence may therefore meet the one before it.)
struct Turn {
  std::mutex mtx;
  hipStream_t first = nullptr;
  bool used = false, several = false;
  hipEvent_t event = nullptr;
  bool recorded = false;
};
Turn g_turns[16];

// of the current device; 0: unknown
int compute_units() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return cus;
}

}  // namespace

}  // namespace tfcc_rocm

using namespace tfcc_rocm;

extern "C" {

size_t tfcc_rocm_lstm_sequence_workspace(unsigned batch, unsigned units, unsigned directions) {
  return lstm_plan::workspace_bytes(batch, units, directions, compute_units());
}

static int sequence(void* stream, const tfcc_rocm_lstm_sequence_desc* q, bool spread) {
  TFCC_REQUIRE(q != nullptr, "lstm_sequence: null argument");
  const size_t need = tfcc_rocm_lstm_sequence_workspace(q->batch, q->units, q->directions);
  TFCC_REQUIRE(need != 0, "lstm_sequence: 1 to 16 rows, 1 to 1024 units, 1 or 2 directions and a CU for eight units of each, got %u, %u, %u",
               q->batch, q->units, q->directions);
  TFCC_REQUIRE(q->seq >= 1 && q->seq < 0xfffffff0u, "lstm_sequence: %u steps", q->seq);
  TFCC_REQUIRE(q->workspace && (uintptr_t)q->workspace % 8 == 0 && q->workspace_bytes >= need,
               "lstm_sequence: the workspace needs %zu bytes", need);
  SequenceParams p{};
  for (unsigned d = 0; d < q->directions; ++d) {
    TFCC_REQUIRE(q->x[d] && q->kernel[d] && q->bias[d] && q->h0[d] && q->c0[d] && q->out[d] && q->h[d] && q->c[d],
                 "lstm_sequence: null operand");
    p.s[d] = Sequence{q->x[d], q->kernel[d], q->bias[d], q->h0[d], q->c0[d], q->out[d], q->h[d], q->c[d], q->backward[d]};
  }
  p.seq = q->seq; p.batch = q->batch; p.units = q->units; p.directions = q->directions;
  p.forget = q->forget;
  p.rowsPerGroup = lstm_plan::rows_of_xcd(q->batch, q->units, q->directions, compute_units());
  if (q->seq > kStepMask - 2) p.rowsPerGroup = 0;  // (the words' number has 28 bits)
  p.spread = spread;
  p.groups = p.rowsPerGroup ? (q->batch + p.rowsPerGroup - 1) / p.rowsPerGroup : 0;
  p.words = static_cast<unsigned*>(q->workspace);
  p.failed = reinterpret_cast<unsigned*>(static_cast<char*>(q->workspace) + need - 64);
  p.waitTicks = (unsigned long long)q->wait_us * 100;  // of the 100 MHz clock
  int dev = 0;
  TFCC_HIP_CHECK(hipGetDevice(&dev));
  TFCC_REQUIRE(dev >= 0 && dev < 16, "device index %d", dev);
  hipStream_t s = as_stream(stream);
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capturing) != hipSuccess) (void)hipGetLastError();  // the null stream beside a capture: it is not captured
  if (capturing != hipStreamCaptureStatusNone) {
    p.rowsPerGroup = 0;  // replays are not ordered among one another; two of the first form fit side by side up to 512 units
    return launch_units(s, p);
  }
  Turn& turn = g_turns[dev];
  std::lock_guard<std::mutex> lk(turn.mtx);
  if (!turn.used) turn.first = s;
  turn.several = turn.several || (turn.used && turn.first != s) || s == hipStreamPerThread;
  turn.used = true;
  if (!turn.several) return launch_units(s, p);
  if (turn.event == nullptr) TFCC_HIP_CHECK(hipEventCreateWithFlags(&turn.event, hipEventDisableTiming));
  // (what cannot be waited for or recorded is done without: the sequences may then meet, and still end)
  if (turn.recorded && hipStreamWaitEvent(s, turn.event, 0) != hipSuccess) (void)hipGetLastError();
  const int status = launch_units(s, p);
  turn.recorded = hipEventRecord(turn.event, s) == hipSuccess;
  if (!turn.recorded) (void)hipGetLastError();
  return status;
}

int tfcc_rocm_lstm_sequence_f32(void* stream, const tfcc_rocm_lstm_sequence_desc* q) { return sequence(stream, q, false); }
int tfcc_rocm_lstm_sequence_f32_spread(void* stream, const tfcc_rocm_lstm_sequence_desc* q) { return sequence(stream, q, true); }

}  // extern "C"
