// fp32 matrix product on the bf16 matrix cores: every operand is split into three bf16 numbers that add up to it exactly.
//
// The fp32 matrix ops deliver 157 TFLOP/s, the bf16 ones sixteen times that.  A float's 24 bits are three bf16 numbers of
// eight: x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1, all exact (rounding to nearest halves what is left each time, so
// the third has room for the rest).  Of the nine products of pieces the six largest are formed, a2 b0, a1 b0, a0 b0, a1 b1,
// a0 b1, a0 b2.  The three left out come to 2^-24.2 of a b at most (2^-28 on the average, with either sign), so a product
// by itself may be off by one unit in the last place instead of half a one.
//
// a0 b0 has an accumulator of its own.  Its products have sixteen bits, so their sums are exact or nearly so, and the
// five small terms meet in a second one 2^8 below; the two are added once, at the end.  (All six in one accumulator take half
// the registers, but there the small terms are rounded at the size of the result: fewer roundings than in the fp32 ops for
// dense operands, which take two k at a time, but more for sparse ones, where an fp32 op adds one product or none.)
// Against 64 bits, relative 2-norm in 1e-8, here, in one accumulator, and with the fp32 ops:
//                  4096^3, 128 x 256 tiles   1024 x 1024 x 2048, 64 x 64   2048^3, 128 x 128 (always in two)
//   normal           40   101   115             13.4   35.2   57.5            27.2   80.9
//   relu(normal)     32    94    81             10.6   33.7   40.5            21.6   57.7
//   10 % dense       14    64    36              6.6   24.5   18.5             9.6   25.7
//   2 % dense         6.4  34    16              5.1   13.8    8.9             4.8   11.7
//   one in a row      2.6   5.4   2.5            2.6    5.4    2.5             2.6    2.5
//
// What the split cannot represent is found and done again.  Infinities, NaN and values that round up to infinity make the
// results they enter NaN or infinite; operands below 2^-109 leave bits of x2 outside bf16's range, which matters next to a very
// large partner or in a very small result; products below 2^-126 round where the fp32 op would not.  So every thread keeps the
// largest magnitude it split of A and of B (one instruction for two values), and looks at its results: those that are not
// finite are formed with the fp32 matrix ops; those below 2^-64 are right if their row or column holds nothing but zeros,
// which the magnitudes tell; about the others the smallest operands of their rows and columns decide, for which those of a few
// results, which happens by chance (a sum that cancels to zero, in one product of ten), are read once more, and all of the
// tile's if there are many (sparse operands on both sides) or a magnitude was 2^30 or more.
//
// What that costs, us, in order, on one card: normal operands; one row of zeros; the last quarter of the rows; one value in a
// hundred in both operands; one value of 2^31; one NaN; two results that cancel; and any operands on the fp32 ops:
//   4096^3, 128 x 256 tiles        602   602   589   583   683   1459   595   910
//   2048^3, 128 x 128               90    91    89   101   110    296    94   120   (two K groups, as the next)
//   1024 x 768 x 3072, 128 x 128    36    38    36    46    45    112    38    40
//   1024 x 1024 x 2048, 64 x 64     30    31    30    45    47    106    31    33
//
// Two kernels.  What they have in common is that vector instructions run under bf16 matrix ops: up to six of them between
// two of 32 cycles cost next to nothing, if they stand there; a wavefront that issues matrix ops back to back keeps the
// others' vector instructions waiting.  The order of both loops is therefore written down.
#include <type_traits>

#include "common.hpp"
#include "lds_dma.hpp"
#include "sgemm_params.hpp"
#include "sgemm_split_plan.hpp"

namespace tfcc_rocm {

using sgemm_detail::SgemmParams;

namespace {

typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// a byte offset that fails the range check of any operand here (below 2^31 bytes, the dispatcher sees to it), also with a
// tile's rows of one added
constexpr unsigned kOutside = 0x80000000u;

// magnitudes, as their bits: infinity, 2^30, 2^-64, 2^-90
constexpr unsigned kInfinite = 0x7f800000u, kLarge = 0x4e800000u, kSmall = 0x1f800000u, kVerySmall = 0x12800000u;

// f(FROM), f(FROM + 1), ..., f(TO - 1) with the index a constant
template <int FROM, int TO, class F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (FROM < TO) {
    f(std::integral_constant<int, FROM>{});
    each<FROM + 1, TO>(f);
  }
}

// V (four or eight) consecutive k of a row or column on their way to three operand pieces, in 6 V instructions that are dealt
// out between the matrix ops, few of which need a result of the three before them.
template <int V>
struct Splitting {
  unsigned piece[3][V / 2];
  float e[4];
};

// the piece that is complete, and can be written to LDS, a little before this operation; or -1
template <int V>
constexpr int written(int op) { return op == V + 2 ? 0 : op == V / 2 * 7 + 2 ? 1 : op == 6 * V - 1 ? 2 : -1; }

template <int V, int op>
__device__ __forceinline__ void split_op(float (&x)[V], Splitting<V>& t, float& largest) {
  if constexpr (op < V && op % 2 == 1) {  // (a conversion between two of the magnitudes, which depend on one another)
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(largest) : "v"(x[op - 1]), "v"(x[op]));
  } else {
    // V / 2 conversions, then twice: V widened and subtracted, four at a time, and V / 2 conversions
    constexpr int H = V / 2, o = op < V ? op / 2 : op - H, stage = o / (5 * H), in = o % (5 * H);
    if constexpr (in < H) {
      unsigned pair = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f{x[2 * in], x[2 * in + 1]}), v2bf));
      asm("" : "+v"(pair));  // or the compiler works parts of it out again where they are used
      t.piece[stage][in] = pair;
    } else {
      constexpr int v = (in - H) / 8 * 4 + (in - H) % 4;  // the value
      const unsigned p = t.piece[stage][v / 2];
      if constexpr ((in - H) % 8 < 4) t.e[v & 3] = __builtin_bit_cast(float, v & 1 ? p & 0xffff0000u : p << 16);
      else x[v] -= t.e[v & 3];
    }
  }
}

// the six terms of a product: the pieces of A and of B
constexpr int kTermA[6] = {2, 1, 0, 1, 0, 0}, kTermB[6] = {0, 0, 0, 1, 1, 2};
__device__ __forceinline__ v16f product(v4u a, v4u b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

__device__ __forceinline__ v4u operand(const unsigned (&x)[4]) { return v4u{x[0], x[1], x[2], x[3]}; }

// A tile of the launch and its operands.
struct Tile {
  unsigned m0, n0, bi;
  const float *A, *B, *bias, *R;
  float* C;
  unsigned bytesA, bytesB;
  bool exists;
};
template <int BM, int BN, bool TRANSB>
__device__ __forceinline__ Tile tile_of(const SgemmParams& p) {
  Tile t;
  // consecutive workgroup ids land on different XCDs: hand each XCD a contiguous run of tiles
  const unsigned xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, L = xcd * p.chunk + slot;
  t.exists = slot < p.chunk && L < p.tilesTotal;
  t.bi = udiv_apply(L, p.perBatchMagic, p.perBatchShift);
  const unsigned w = L - t.bi * p.tilesM * p.tilesN, band = 4u * p.tilesN, b = udiv_apply(w, p.bandMagic, p.bandShift);
  const unsigned rows = min(4u, p.tilesM - b * 4u), r = w - b * band, q = rows == 4u ? r >> 2 : r / rows;
  t.m0 = (b * 4u + (r - q * rows)) * BM;
  t.n0 = q * BN;
  const unsigned bo = udiv_apply(t.bi, p.innerMagic, p.innerShift), bn = t.bi - bo * p.batchInner;
  t.A = p.A + (size_t)bo * p.strideA + (size_t)bn * p.innerA;
  t.B = p.B + (size_t)bo * p.strideB + (size_t)bn * p.innerB;
  t.bias = p.bias;
  t.C = p.C + (size_t)bo * p.strideC + (size_t)bn * p.innerC;
  if (p.groups) {  // selects, not indexing: the argument block stays in scalar registers
    t.A = p.A;
    t.B = t.bi == 0 ? p.groupB[0] : t.bi == 1 ? p.groupB[1] : t.bi == 2 ? p.groupB[2] : p.groupB[3];
    t.bias = t.bi == 0 ? p.groupBias[0] : t.bi == 1 ? p.groupBias[1] : t.bi == 2 ? p.groupBias[2] : p.groupBias[3];
    t.C = t.bi == 0 ? p.groupC[0] : t.bi == 1 ? p.groupC[1] : t.bi == 2 ? p.groupC[2] : p.groupC[3];
  }
  t.R = p.residual ? p.residual + (size_t)t.bi * p.strideR : nullptr;  // dense, flat batch
  t.bytesA = ((p.M - 1) * p.lda + p.K) * 4u;
  t.bytesB = TRANSB ? ((p.N - 1) * p.ldb + p.K) * 4u : ((p.K - 1) * p.ldb + p.N) * 4u;
  return t;
}

// The smallest of the sixteen lanes' values, in all of them.
__device__ __forceinline__ unsigned least_of_sixteen(unsigned x) {
  x = min(x, (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0xb1, 0xf, 0xf, true));   // quad_perm 1, 0, 3, 2
  x = min(x, (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x4e, 0xf, 0xf, true));   // quad_perm 2, 3, 0, 1
  x = min(x, (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xf, 0xf, true));  // row_half_mirror
  return min(x, (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x140, 0xf, 0xf, true));  // row_mirror
}

// The smallest magnitude other than zero in every one of `rows` (at most ROWS) rows of `n` floats, by T threads, or of all of
// them in every one of `n` (at most COLS) columns, as twice its bits less one: zero counts as the largest.  (Loaded as whole
// numbers: a bit_cast of a vector's element reads its first one.)
template <int ROWS, int T>
__device__ __forceinline__ void least_of_rows(const float* x, unsigned rows, unsigned n, unsigned ld, unsigned* least) {
  constexpr int EACH = ROWS * 16 / T, CHUNKS = 8 / EACH;  // sixteen lanes to a row
  const __amdgpu_buffer_rsrc_t d =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0, (int)(((rows - 1) * ld + n) * 4u), 0x00020000);
  const unsigned lane = threadIdx.x & 15, row = threadIdx.x >> 4;
  unsigned smallest[EACH];
#pragma unroll
  for (int u = 0; u < EACH; ++u) smallest[u] = ~0u;
  for (unsigned first = 4 * lane; first < n; first += 64 * CHUNKS) {
    v4u v[EACH][CHUNKS];
#pragma unroll
    for (int u = 0; u < EACH; ++u)
#pragma unroll
      for (int k = 0; k < CHUNKS; ++k) {
        const unsigned r = row + u * (T / 16), c = first + 64 * k;
        v[u][k] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(d, c < n && r < rows ? (r * ld + c) * 4u : kOutside, 0, 0));
      }
#pragma unroll
    for (int u = 0; u < EACH; ++u)
#pragma unroll
      for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
        for (unsigned e = 0; e < 4; ++e) smallest[u] = min(smallest[u], first + 64 * k + e < n ? (v[u][k][e] << 1) - 1u : ~0u);
  }
#pragma unroll
  for (int u = 0; u < EACH; ++u) {
    const unsigned value = least_of_sixteen(smallest[u]);
    if (lane == 0) least[row + u * (T / 16)] = value;
  }
}
template <int COLS, int T>
__device__ __forceinline__ void least_of_columns(const float* x, unsigned rows, unsigned n, unsigned ld, unsigned* least) {
  const __amdgpu_buffer_rsrc_t d =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0, (int)(((rows - 1) * ld + n) * 4u), 0x00020000);
  constexpr int STEP = T / (COLS / 4);  // rows at a time
  const unsigned c = 4 * (threadIdx.x % (COLS / 4));
  v4u smallest = {~0u, ~0u, ~0u, ~0u};
  for (unsigned r = threadIdx.x / (COLS / 4); r < rows; r += 8 * STEP) {
    v4u v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      v[u] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(d, c < n && r + u * STEP < rows ? ((r + u * STEP) * ld + c) * 4u : kOutside, 0, 0));
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) smallest[e] = min(smallest[e], (v[u][e] << 1) - 1u);
  }
#pragma unroll
  for (unsigned e = 0; e < 4; ++e)
    if (c + e < n) __hip_atomic_fetch_min(least + c + e, smallest[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// What a workgroup finds out about its tile when a result or an operand looks as if the split may have got something wrong.
constexpr unsigned kMostListed = 32;
template <int BM, int BN>
struct Findings {
  unsigned count, at[kMostListed];  // results below 2^-64: row of the tile * 256 + column
  unsigned largest[BM + BN];        // the largest magnitude of every row of A, then of every column of B, as its bits
  unsigned least[BM + BN];          // the smallest but zero, as twice its bits less one, of those that were asked for
};

// Whether there are results in the tile that have to be formed again with the fp32 matrix ops, and which of the thread's:
// a bit of `again` for each of its BLOCKS x 16.  value(block, i): one of them; where(block, i, row, column): its place in the
// tile.  `suspicious`: one of them is not finite or below 2^-64, or the thread has split a value of 2^30 or more.  raise(): puts
// the magnitudes that the thread has split into `largest`.
// A result that is not finite is formed again.  One of a row or a column of zeros is right, and raise() leaves those outside the
// matrix at zero, so that they are never listed: a listed one's row and column are read.  Others below 2^-64, and those that a
// value of 2^30 or more enters, are formed again if their own row or column has a value that is too small for them.  For a few
// such results their rows and columns are searched for it, for many, or next to a large value, all of the tile's.  Whether
// a result is formed again therefore depends on its own row and column alone.
template <int BM, int BN, int T, bool TRANSB, int BLOCKS, class Value, class Where, class Raise>
__device__ __forceinline__ bool split_failed(const SgemmParams& p, const Tile& t, bool suspicious, Findings<BM, BN>& found,
                                             unsigned (&again)[BLOCKS], Value&& value, Where&& where, Raise&& raise) {
  if (!__syncthreads_or(suspicious)) return false;
  if (threadIdx.x == 0) found.count = 0;
  for (unsigned i = threadIdx.x; i < BM + BN; i += T) {
    found.largest[i] = 0;
    found.least[i] = ~0u;
  }
  __syncthreads();
  raise();
  __syncthreads();
  bool large = false;
  for (unsigned i = threadIdx.x; i < BM + BN; i += T) large = large || found.largest[i] >= kLarge;
  unsigned any = 0;
  // (without branches: 64 results are looked at in 1 us)
  each<0, BLOCKS>([&](auto b) __attribute__((always_inline)) {
    unsigned wrong = 0, small = 0;
    each<0, 16>([&](auto i) __attribute__((always_inline)) {
      unsigned row, col;
      where(b, i, row, col);
      const unsigned size = __builtin_bit_cast(unsigned, value(b, i)) & 0x7fffffffu;
      wrong |= (unsigned)(size >= kInfinite) << i;
      small |= (unsigned)((size < kSmall) & (found.largest[row] != 0) & (found.largest[BM + col] != 0)) << i;
    });
    again[b] = wrong;
    any |= wrong;
    for (; small != 0; small &= small - 1) {
      unsigned row, col;
      where(b, __builtin_ctz(small), row, col);
      const unsigned at = atomicAdd(&found.count, 1u);
      if (at < kMostListed) found.at[at] = row << 8 | col;
    }
  });
  large = __syncthreads_or(large) != 0;
  if (large || found.count > kMostListed) {
    const unsigned rows = min((unsigned)BM, p.M - t.m0), cols = min((unsigned)BN, p.N - t.n0);
    least_of_rows<BM, T>(t.A + (size_t)t.m0 * p.lda, rows, p.K, p.lda, found.least);
    if constexpr (TRANSB) least_of_rows<BN, T>(t.B + (size_t)t.n0 * p.ldb, cols, p.K, p.ldb, found.least + BM);
    else least_of_columns<BN, T>(t.B + t.n0, p.K, cols, p.ldb, found.least + BM);
  } else {
    for (unsigned i = 0; i < found.count; ++i) {
      const unsigned row = found.at[i] >> 8, col = found.at[i] & 255u;
      unsigned x = ~0u, y = ~0u;
      for (unsigned k = threadIdx.x; k < p.K; k += T) {
        const float ofA = t.A[(size_t)(t.m0 + row) * p.lda + k];
        const float ofB = TRANSB ? t.B[(size_t)(t.n0 + col) * p.ldb + k] : t.B[(size_t)k * p.ldb + t.n0 + col];
        x = min(x, (__builtin_bit_cast(unsigned, ofA) << 1) - 1u);
        y = min(y, (__builtin_bit_cast(unsigned, ofB) << 1) - 1u);
      }
      x = least_of_sixteen(x);
      y = least_of_sixteen(y);
      if ((threadIdx.x & 15) == 0) {
        __hip_atomic_fetch_min(&found.least[row], x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_fetch_min(&found.least[BM + col], y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
  }
  if (!large && found.count == 0) return __syncthreads_or(any != 0) != 0;
  __syncthreads();
  each<0, BLOCKS>([&](auto b) __attribute__((always_inline)) {
    each<0, 16>([&](auto i) __attribute__((always_inline)) {
      unsigned row, col;
      where(b, i, row, col);
      const unsigned size = __builtin_bit_cast(unsigned, value(b, i)) & 0x7fffffffu;
      const bool candidate = (size < kSmall) | (found.largest[row] >= kLarge) | (found.largest[BM + col] >= kLarge);
      const int x = (int)(found.least[row] >> 24) - 127, y = (int)(found.least[BM + col] >> 24) - 127;  // exponents
      again[b] |= (unsigned)(candidate & ((x < -100) | (y < -100) | ((x + y < -100) & (size < kVerySmall)))) << i;
    });
    any |= again[b];
  });
  return __syncthreads_or(any != 0) != 0;
}

// ---- large products ------------------------------------------------------------------------------------------------------
// A workgroup of WGM x WGN wavefronts, a wavefront (32 MI) x (32 NI) outputs.  K goes in slabs of sixteen, one matrix op
// deep: a thread loads four or eight values of a row of A and eight of a column of B and splits them on the way from its
// registers to LDS, once for the workgroup; the wavefronts read the pieces in operand order.
//
// Bound by power, the matrix cores and the splitting: 4096^3 in 128 x 256 tiles 910 -> 602 us, 228 TFLOP/s (214 to 228 by the
// card); the matrix ops alone, from registers on the same operands, sustain 302.  Times against 623 on another card:
// (128 x 128 tiles, two to a CU, split four values to six
// matrix ops' worth instead of three: 669 us.  256 x 256 tiles, two values: 600, but there are registers for one
// accumulator only; with a block's six terms summed from zero, smallest first, and then added to it 635, and one
// product in a row still 3.5e-8.  A wavefront for each SIMD on 128 x 128, more slabs on their way, two K groups
// of such tiles: all slower.  What is left of a value beside its piece as one dot product of pieces with -1, two instructions
// fewer for each value: the dot products run in the matrix cores, 675 against 634.)
//
// KG = 2: two such groups of wavefronts have a tile, every other slab each, and meet in LDS; for products with one tile to a CU
// at most, where a wavefront for each SIMD has nothing beside it while it waits (sgemm_split_plan.hpp).
template <int BM, int BN>
struct SharedLayout {
  // [piece][eight k][row or column] of 16 bytes; 64 bytes between the halves of k put a thread pair's writes on
  // different banks
  static constexpr int HALF_A = BM * 16 + 64, HALF_B = BN * 16 + 64, PIECE_A = 2 * HALF_A, PIECE_B = 2 * HALF_B,
                       STAGE = 3 * (PIECE_A + PIECE_B);
};

template <int MI, int NI, int WGM, int WGN, int KG, bool TRANSB>
__global__ __launch_bounds__(64 * WGM * WGN * KG, 2) void sgemm_split_kernel(const SgemmParams p) {
  constexpr int BM = 32 * MI * WGM, BN = 32 * NI * WGN, BK = 16, T = 64 * WGM * WGN;
  constexpr int VA = BM * BK / T, VB = BN * BK / T, OPS_A = 6 * VA, OPS = OPS_A + 6 * VB;  // values per thread
  static_assert((VA == 4 || VA == 8) && VB == 8, "a thread has four or eight values of A and eight of B");
  using L = SharedLayout<BM, BN>;
  constexpr int STAGE = L::STAGE;

  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ Findings<BM, BN> found;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int grp = KG == 1 ? 0 : wave / (WGM * WGN), wv = wave - grp * WGM * WGN;
  const int wm = wv / WGN, wn = wv - wm * WGN;  // wave-uniform
  const int tid = KG == 1 ? threadIdx.x : threadIdx.x % T, lane = tid & 63, lrow = lane & 31, g = lane >> 5;
  unsigned char* const gsm = smem + grp * 3 * STAGE;
  const Tile tile = tile_of<BM, BN, TRANSB>(p);
  if (!tile.exists) return;
  const unsigned m0 = tile.m0, n0 = tile.n0, M = p.M, N = p.N, K = p.K, lda = p.lda, ldb = p.ldb;
  const float *A = tile.A, *B = tile.B;

  // ---- loads.  Rows of A (and of B given transposed): two threads to a row, eight k each, or four, four k each.  B as
  // stored: a thread to a column, eight rows.  Past the operands' ends lie zeros (the range check looks at the lane's offset, so the slab's k
  // is in the descriptor); past the end of a row of A lies the next one, which the last slab masks.
  const int arow = tid / (BK / VA), ak = tid % (BK / VA) * VA;
  const int brow = TRANSB ? tid >> 1 : tid & (BN - 1), bhalf = TRANSB ? tid & 1 : tid / BN;
  const unsigned aOff = m0 + arow < M ? ((m0 + arow) * lda + ak) * 4u : kOutside;
  const unsigned bOff = n0 + brow >= N ? kOutside : TRANSB ? ((n0 + brow) * ldb + 8 * bhalf) * 4u : (8 * bhalf * ldb + n0 + brow) * 4u;
  const unsigned slabs = (K + KG * BK - 1) / (KG * BK);  // of every K group
  auto firstK = [&](unsigned s) { return (s * KG + grp) * (unsigned)BK; };
  struct Raw { float a[VA], b[VB]; };
  // the operand from its k `k0` on, `step` bytes to a k: 32-bit scalar arithmetic (a 64-bit comparison would be made on the
  // vector unit, and the descriptor then read back lane by lane)
  auto descriptor = [&](const float* base, unsigned k0, unsigned step, unsigned bytes) {
    const unsigned skip = k0 < K ? k0 * step : 0u;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base) + skip / 4, 0, k0 < K ? (int)(bytes - skip) : 0, 0x00020000);
  };
  // one of the loads of slab s, A's first
  constexpr int LOADS_A = VA / 4, LOADS = LOADS_A + (TRANSB ? 2 : 8);
  auto load = [&](Raw& r, unsigned s, int which) __attribute__((always_inline)) {
    const unsigned k0 = firstK(s);
    auto quad = [&](float* x, __amdgpu_buffer_rsrc_t d, unsigned off) __attribute__((always_inline)) {
      const v4f v = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(d, off, 0, 0));
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = v[e];
    };
    const int ofB = which - LOADS_A;
    if (ofB < 0)
      quad(r.a + 4 * which, descriptor(A, k0, 4u, tile.bytesA), aOff + 16 * which);
    else if (TRANSB)
      quad(r.b + 4 * ofB, descriptor(B, k0, 4u, tile.bytesB), bOff + 16 * ofB);
    else  // (a scalar offset is not range-checked)
      r.b[ofB] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(descriptor(B, k0, ldb * 4u, tile.bytesB),
                                                                               bOff + ofB * ldb * 4u, 0, 0));
  };
  auto mask = [&](Raw& r, unsigned s) {  // the slab in which K ends, or one behind it
    const int left = (int)K - (int)firstK(s);
#pragma unroll
    for (int e = 0; e < VA; ++e) r.a[e] = ak + e < left ? r.a[e] : 0.f;
#pragma unroll
    for (int e = 0; e < VB; ++e) r.b[e] = 8 * bhalf + e < left ? r.b[e] : 0.f;
  };
  float largestA = 0.f, largestB = 0.f;
  unsigned char* const aTo = gsm + ak / 8 * L::HALF_A + arow * 16 + ak % 8 * 2;
  unsigned char* const bTo = gsm + 3 * L::PIECE_A + bhalf * L::HALF_B + brow * 16;

  v16f main[MI][NI], rest[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) main[i][j] = rest[i][j] = v16f{};

  const unsigned char* const aFrom = gsm + g * L::HALF_A + (wm * 32 * MI + lrow) * 16;
  const unsigned char* const bFrom = gsm + 3 * L::PIECE_A + g * L::HALF_B + (wn * 32 * NI + lrow) * 16;
  Raw raw;
  Splitting<VA> ofA;
  Splitting<VB> ofB;
  v4u a[3][MI], b[3][NI];
  // The instructions that split a thread's values, A's, then B's.  Each piece is written when it is there, a while before
  // the next: three writes in a row hold the wavefront up (by a tenth, in 256 x 256 tiles).
  auto splitOp = [&](Raw& r, unsigned stage, auto op) __attribute__((always_inline)) {
    if constexpr (op < OPS_A) {
      split_op<VA, op>(r.a, ofA, largestA);
      constexpr int w = written<VA>(op);
      if constexpr (w >= 0 && VA == 8)
        *reinterpret_cast<v4u*>(aTo + stage + w * L::PIECE_A) = v4u{ofA.piece[w][0], ofA.piece[w][1], ofA.piece[w][VA / 2 - 2], ofA.piece[w][VA / 2 - 1]};
      else if constexpr (w >= 0)
        *reinterpret_cast<v2u*>(aTo + stage + w * L::PIECE_A) = v2u{ofA.piece[w][0], ofA.piece[w][1]};
    } else {
      split_op<VB, op - OPS_A>(r.b, ofB, largestB);
      constexpr int w = written<VB>(op - OPS_A);
      if constexpr (w >= 0)
        *reinterpret_cast<v4u*>(bTo + stage + w * L::PIECE_B) = v4u{ofB.piece[w][0], ofB.piece[w][1], ofB.piece[w][2], ofB.piece[w][3]};
    }
  };
  auto readA = [&](int i, int j, unsigned stage) __attribute__((always_inline)) {
    a[i][j] = *reinterpret_cast<const v4u*>(aFrom + stage + i * L::PIECE_A + j * 512);
  };
  auto readB = [&](int i, int j, unsigned stage) __attribute__((always_inline)) {
    b[i][j] = *reinterpret_cast<const v4u*>(bFrom + stage + i * L::PIECE_B + j * 512);
  };

  // ---- slabs 0 and 1 in LDS, slab 2 on its way, the first operands in registers
  Raw ahead[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int w = 0; w < LOADS; ++w) {
      load(ahead[s], s, w);
      __builtin_amdgcn_sched_barrier(0);  // in the order of the loop, whose waits count on it
    }
#pragma unroll
  for (int w = 0; w < LOADS; ++w) {
    load(raw, 2, w);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (firstK(s) + BK > K) mask(ahead[s], s);
    each<0, OPS>([&](auto o) __attribute__((always_inline)) { splitOp(ahead[s], s * STAGE, o); });
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MI; ++i) readA(2, i, 0);
#pragma unroll
  for (int j = 0; j < NI; ++j) readB(0, j, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < MI; ++i) readA(1, i, 0);
#pragma unroll
  for (int j = 0; j < NI; ++j) readB(1, j, 0);
  __builtin_amdgcn_sched_barrier(0);

  // ---- A slab is six terms of MI NI matrix ops.  Their order, a2 b0, a1 b0, a0 b0, a1 b1, a0 b1, a0 b2, lets every operand
  // be read again, for the next slab, well before its first use there; only a0 and b2 are read in their own slab.  Between
  // the matrix ops the values of the slab after the next are split and written, and the one behind that is asked for.  Of
  // the three stages one is read, one is complete, one is written, so a single barrier in a slab is enough.
  constexpr int PT = MI * NI, TOTAL = 6 * PT, SPREAD = 5 * PT;  // SPREAD: matrix ops that the splitting is dealt out behind
  unsigned st0 = 0, st1 = STAGE, st2 = 2 * STAGE;               // stages of slabs s, s + 1, s + 2
  for (unsigned s = 0; s < slabs; ++s) {
    if (firstK(s + 2) + BK > K) mask(raw, s + 2);
    each<0, TOTAL>([&](auto mc) __attribute__((always_inline)) {
      constexpr int m = mc, t = m / PT, i = m % PT / NI, j = m % NI;
      v16f& sum = t == 2 ? main[i][j] : rest[i][j];
      sum = product(a[kTermA[t]][i], b[kTermB[t]][j], sum);
      if (m == 0) __syncthreads();
      if (m >= 1 && m <= MI) readA(0, m - 1, st0);
      if (m > MI && m <= MI + NI) readB(2, m - MI - 1, st0);
      constexpr int from = m < SPREAD ? m * OPS / SPREAD : OPS, to = m < SPREAD ? (m + 1) * OPS / SPREAD : from;
      each<from, to>([&](auto o) __attribute__((always_inline)) {
        splitOp(raw, st2, o);
        if constexpr (o == OPS_A + 3) load(raw, s + 3, 0);
        if constexpr (o == OPS_A + 7 && LOADS_A == 2) load(raw, s + 3, 1);
      });
      if (m >= SPREAD && m - SPREAD < (LOADS - LOADS_A) / 2) {
        load(raw, s + 3, LOADS_A + 2 * (m - SPREAD));
        load(raw, s + 3, LOADS_A + 1 + 2 * (m - SPREAD));
      }
      if (m >= 2 * PT && m < 2 * PT + MI) readA(2, m - 2 * PT, st1);
      if (m >= 3 * PT && m < 3 * PT + NI) readB(0, m - 3 * PT, st1);
      if (m >= 4 * PT && m < 4 * PT + MI) readA(1, m - 4 * PT, st1);
      if (m >= 5 * PT && m < 5 * PT + NI) readB(1, m - 5 * PT, st1);
      __builtin_amdgcn_sched_barrier(0);
    });
    const unsigned done = st0;
    st0 = st1;
    st1 = st2;
    st2 = done;
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) main[i][j][r] += rest[i][j][r];

  // ---- the K groups' sums meet in LDS; each finishes its share of the rows
  constexpr int MO = MI / KG;
  v16f out[MO][NI];
  if constexpr (KG == 1) {
#pragma unroll
    for (int i = 0; i < MO; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) out[i][j] = main[i][j];
  } else {
    static_assert(KG == 2 && MI == 2, "two K groups, a block of rows for each");
    __syncthreads();
    v4f* const meeting = reinterpret_cast<v4f*>(smem) + wv * NI * 4 * 64 + lane;  // [receiving group][wavefront][quad of values][lane]
    constexpr int HALF = WGM * WGN * NI * 4 * 64;
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        v4f v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = grp == 0 ? main[1][j][4 * c + e] : main[0][j][4 * c + e];
        meeting[(1 - grp) * HALF + (4 * j + c) * 64] = v;
      }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const v4f v = meeting[grp * HALF + (4 * j + c) * 64];
#pragma unroll
        for (int e = 0; e < 4; ++e)  // (a sum of two: the same bits either way round)
          out[0][j][4 * c + e] = (grp == 0 ? main[0][j][4 * c + e] : main[1][j][4 * c + e]) + v[e];
      }
  }

  // ---- what the split may have got wrong
  const unsigned rowBase = m0 + wm * MI * 32 + grp * MO * 32, colBase = n0 + wn * NI * 32;
  float notFinite = 0.f, low = 1.f;
#pragma unroll
  for (int i = 0; i < MO; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        notFinite = fmaf(out[i][j][r], 0.f, notFinite);
        low = fminf(low, __builtin_fabsf(out[i][j][r]));
      }
  if (rowBase + 32 * MO > M || colBase + 32 * NI > N) {  // the zeros outside the matrix do not count
    low = 1.f;
#pragma unroll
    for (int i = 0; i < MO; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (rowBase + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3) < M && colBase + 32 * j + lrow < N)
            low = fminf(low, __builtin_fabsf(out[i][j][r]));
  }
  auto raise = [&]() {
    __hip_atomic_fetch_max(&found.largest[arow], __builtin_bit_cast(unsigned, largestA), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_max(&found.largest[BM + brow], __builtin_bit_cast(unsigned, largestB), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto value = [&](auto block, auto r) __attribute__((always_inline)) -> float {
    const float v = out[block / NI][block % NI][(int)r];  // (a copy: a bit_cast of a vector's element reads its first one)
    return v;
  };
  auto where = [&](int block, int r, unsigned& row, unsigned& col) __attribute__((always_inline)) {
    row = wm * MI * 32 + grp * MO * 32 + 32 * (block / NI) + 8 * (r >> 2) + 4 * g + (r & 3);
    col = wn * NI * 32 + 32 * (block % NI) + lrow;
  };
  unsigned again[MO * NI];
  const bool suspicious = notFinite != 0.f || low < 0x1p-64f || largestA >= 0x1p30f || largestB >= 0x1p30f;
  if (split_failed<BM, BN, T * KG, TRANSB, MO * NI>(p, tile, suspicious, found, again, value, where, raise)) {
#pragma unroll
    for (int i = 0; i < MO; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        if (!__any(again[i * NI + j] != 0)) continue;
        const unsigned arow = rowBase + 32 * i + lrow, bcol = colBase + 32 * j + lrow;
        v16f sum = {};
        for (unsigned k = 0; k < K; k += 32) {
          float x[16], y[16];
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const unsigned kk = k + 2 * e + g;
            x[e] = kk < K && arow < M ? A[(size_t)arow * lda + kk] : 0.f;
            y[e] = kk < K && bcol < N ? TRANSB ? B[(size_t)bcol * ldb + kk] : B[(size_t)kk * ldb + bcol] : 0.f;
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], y[e], sum, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) out[i][j][r] = again[i * NI + j] >> r & 1 ? sum[r] : out[i][j][r];
      }
  }

  // ---- tile store: + bias, + residual, GELU; rows past M and columns past N fail the range check
  const bool inside = rowBase < M && colBase < N;
  const unsigned ldc = p.ldc, rows = inside ? min(M - rowBase, 32u * MO) : 1u;
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(tile.C + (size_t)rowBase * ldc + colBase, 0,
                                                                      (int)(((rows - 1) * ldc + N - colBase) * 4u), 0x00020000);
  const float* R = tile.R ? tile.R + (size_t)rowBase * N + colBase : nullptr;
  float bv[NI];
  unsigned to[NI], from[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const bool in = colBase + 32 * j + lrow < N;
    bv[j] = tile.bias && in ? tile.bias[colBase + 32 * j + lrow] : 0.f;
    to[j] = in ? ((4 * g) * ldc + 32 * j + lrow) * 4u : kOutside;
    from[j] = in ? ((4 * g) * N + 32 * j + lrow) * 4u : kOutside;
  }
  auto store_all = [&](bool residual, bool gelu) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rr =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(R), 0, (int)(((rows - 1) * N + N - colBase) * 4u), 0x00020000);
#pragma unroll
    for (int i = 0; i < MO; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const unsigned row = 32 * i + 8 * (r >> 2) + (r & 3);
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          float v = out[i][j][r] + bv[j];
          if (residual) v += __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rr, from[j] + row * N * 4u, 0, 0));
          // same expression as the stand-alone GELU kernel, so that fusing changes no bit
          if (gelu) v = gelu_erf_f32(v);
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rc, to[j] + row * ldc * 4u, 0, 0);
        }
      }
  };
  if (inside) {
    if (p.act == 1) store_all(R != nullptr, true);
    else store_all(R != nullptr, false);
  }
}

// ---- products of a few dozen to a few hundred tiles ------------------------------------------------------------------
// KG wavefronts own 64 x 64 outputs; wavefront q sums the slabs of 32 k q, q + KG, ... for all of them.  Copies go straight to
// a ring in LDS that belongs to the wavefront, so there is no barrier until the partial tiles meet; a wavefront splits what it
// multiplies by itself, twice the splitting of a 128 x 128 tile shared by four, and the vector unit bounds the loop: eight of
// its instructions to a matrix op, 1250 cycles for the 768 that a step's matrix ops take.  The second accumulator costs it
// nothing, 31.8 us for 1024 x 1024 x 2048 with and without.  (Operands fetched straight to
// registers: the address unit is the bound, 38 us against 33.5 for 1024 x 3072 x 768.)
template <int KG, bool TRANSB>
__global__ __launch_bounds__(64 * KG, 2) void sgemm_split64_kernel(const SgemmParams p) {
  constexpr int BM = 64, BN = 64, BK = 16, STAGES = 2;
  constexpr int A_BYTES = BM * BK * 4, B_BYTES = BK * BN * 4, STAGE = A_BYTES + B_BYTES, COPIES = STAGE / 1024;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ Findings<BM, BN> found;
  const int grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, lrow = lane & 31, g = lane >> 5;
  unsigned char* gsm = smem + grp * STAGES * STAGE;
  const unsigned ldsGroup = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)gsm;
  const Tile tile = tile_of<BM, BN, TRANSB>(p);
  if (!tile.exists) return;
  const unsigned m0 = tile.m0, n0 = tile.n0, M = p.M, N = p.N, K = p.K, lda = p.lda, ldb = p.ldb;

  // ---- copies of 1 KB.  Rows of A (and of B given transposed): 64 bytes each, chunk c of 16 bytes of row r at chunk
  // c ^ (r / 4 & 3); B as stored: k rows of 256 bytes.  The slab's k goes into the descriptor, so what is left of the operand
  // is what a lane's offset is checked against.
  const lds_dma_v4i rsrcA = make_rsrc(tile.A, tile.bytesA), rsrcB = make_rsrc(tile.B, tile.bytesB);
  constexpr int A_COPIES = A_BYTES / 1024, B_COPIES = B_BYTES / 1024;
  unsigned aOff[A_COPIES], bOff[B_COPIES];
#pragma unroll
  for (int u = 0; u < A_COPIES; ++u) {
    const unsigned r = 16 * u + lane / 4, c = (lane & 3) ^ ((r >> 2) & 3);
    aOff[u] = m0 + r < M ? ((m0 + r) * lda + 4 * c) * 4u : kOutside;
    if constexpr (TRANSB) {
      bOff[u] = n0 + r < N ? ((n0 + r) * ldb + 4 * c) * 4u : kOutside;
    } else {
      const unsigned k = 4 * u + lane / 16, col = n0 + 4 * (lane & 15);
      bOff[u] = col < N ? (k * ldb + col) * 4u : kOutside;
    }
  }
  const unsigned slabs = (K + 31) / 32, steps = 2 * ((slabs + KG - 1) / KG);
  auto firstK = [&](unsigned s) { return ((s >> 1) * KG + grp) * 32u + (s & 1u) * BK; };
  auto copy = [&](unsigned s, unsigned stage, int u) __attribute__((always_inline)) {
    const unsigned k0 = firstK(s);
    const bool live = k0 < K, isA = u < A_COPIES;
    const unsigned so = live ? isA || TRANSB ? k0 * 4u : k0 * ldb * 4u : 0u;
    lds_dma_v4i rsrc = isA ? rsrcA : rsrcB;
    const unsigned long long base = (((unsigned long long)(unsigned)rsrc[1] << 32) | (unsigned)rsrc[0]) + so;
    rsrc[0] = (int)(unsigned)base;
    rsrc[1] = (int)(unsigned)(base >> 32);
    rsrc[2] = live ? rsrc[2] - (int)so : 0;
    dma16s(rsrc, ldsGroup + stage * STAGE + u * 1024, isA ? aOff[u] : bOff[u - A_COPIES], 0u);
  };
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
#pragma unroll
    for (int u = 0; u < COPIES; ++u) copy(s, s, u);

  // Lane (c, g) holds rows c and 32 + c, columns 2 c and 2 c + 1, and of a slab the k 8 g .. 8 g + 7.
  struct Raw { float a[2][8], b[2][8]; };
  auto rowValues = [&](float (&x)[8], const unsigned char* image, int row, int h) __attribute__((always_inline)) {
    const v4f v = *reinterpret_cast<const v4f*>(image + row * 64 + (((2 * g + h) ^ ((row >> 2) & 3)) << 4));
#pragma unroll
    for (int e = 0; e < 4; ++e) x[4 * h + e] = v[e];
  };
  // one of the twelve reads of a slab's values (TRANSB: eight): 0 .. 3 are A's
  constexpr int READS = TRANSB ? 8 : 12;
  auto read = [&](Raw& r, unsigned stage, int w) __attribute__((always_inline)) {
    const unsigned char* st = gsm + stage * STAGE;
    if (w < 4) {
      rowValues(r.a[w >> 1], st, 32 * (w >> 1) + lrow, w & 1);
    } else if (TRANSB) {
      rowValues(r.b[(w - 4) >> 1], st + A_BYTES, 2 * lrow + ((w - 4) >> 1), w & 1);
    } else {
      const v2f v = *reinterpret_cast<const v2f*>(st + A_BYTES + (8 * g + w - 4) * 256 + lrow * 8);
      r.b[0][w - 4] = v[0];
      r.b[1][w - 4] = v[1];
    }
  };
  auto mask = [&](Raw& r, unsigned s) __attribute__((always_inline)) {  // the slab in which K ends, or one behind it
    const int left = (int)K - (int)firstK(s) - 8 * g;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        r.a[i][e] = e < left ? r.a[i][e] : 0.f;
        if constexpr (TRANSB) r.b[i][e] = e < left ? r.b[i][e] : 0.f;
      }
  };

  v16f acc[2][2], rest[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = rest[i][j] = v16f{};
  float largest[4] = {};  // of the two rows and of the two columns
  // Two sets of operands: the matrix ops of a step run on one while the next step's values are split into the other, and
  // the values of the step after that are read as their registers fall free.
  Raw raw;
  Splitting<8> a[2][2], b[2][2];
  constexpr int OPS = 48;  // of one of them
  auto splitOp = [&](int set, auto op) __attribute__((always_inline)) {
    constexpr int o = op % OPS, which = op / OPS;
    if constexpr (which < 2) split_op<8, o>(raw.a[which], a[set][which], largest[which]);
    else split_op<8, o>(raw.b[which - 2], b[set][which - 2], largest[which]);
  };
  wait_vmcnt<COPIES*(STAGES - 1)>();
#pragma unroll
  for (int w = 0; w < READS; ++w) read(raw, 0, w);
  if (firstK(0) + BK > K) mask(raw, 0);
  each<0, 4 * OPS>([&](auto o) __attribute__((always_inline)) { splitOp(0, o); });
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the reads of slab 0 have returned
#pragma unroll
  for (int u = 0; u < COPIES; ++u) copy(2, 0, u);
  wait_vmcnt<COPIES*(STAGES - 1)>();
#pragma unroll
  for (int w = 0; w < READS; ++w) read(raw, 1, w);
  auto step = [&](unsigned s, auto set) __attribute__((always_inline)) {
    constexpr int cur = set, nxt = 1 - set;
    // slab s + 1 is in registers, s + 2 in stage `cur`, s + 3 goes to stage `nxt`
    if (firstK(s + 1) + BK > K) mask(raw, s + 1);
    each<0, 24>([&](auto m) __attribute__((always_inline)) {
      constexpr int t = m / 4, i = m / 2 % 2, j = m % 2;
      v16f& sum = t == 2 ? acc[i][j] : rest[i][j];
      sum = product(operand(a[cur][i].piece[kTermA[t]]), operand(b[cur][j].piece[kTermB[t]]), sum);
      each<8 * m, 8 * m + 8>([&](auto o) __attribute__((always_inline)) { splitOp(nxt, o); });
      if constexpr (m == 4) __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the reads of slab s + 1 have returned
      if constexpr (m >= 4 && m <= 7) {
        copy(s + 3, nxt, 2 * (m - 4));
        copy(s + 3, nxt, 2 * (m - 4) + 1);
      }
      if constexpr (m == 8) wait_vmcnt<COPIES>();
      if constexpr (m == 8 || m == 9) read(raw, cur, m - 8);     // A's first block is through with operation 47
      if constexpr (m == 12 || m == 13) read(raw, cur, m - 10);  // its second one with 95
      if constexpr (m == 23) {
#pragma unroll
        for (int w = 4; w < READS; ++w) read(raw, cur, w);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  for (unsigned s = 0; s < steps; s += 2) {  // an even number: two to a slab of 32 k
    step(s, std::integral_constant<int, 0>{});
    step(s + 1, std::integral_constant<int, 1>{});
  }
  wait_vmcnt<0>();
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] += rest[i][j][r];

  // ---- the partial tiles meet: registers 4 c .. 4 c + 3 of block (i, j) as one quad, in the order of i, c, j; wavefront w
  // finishes the quads from w QPW on, rows of two neighbouring columns
  constexpr int QPW = 16 / KG;
  v4f* meetings = reinterpret_cast<v4f*>(smem);
  auto meet = [&](v4f (&sum)[QPW]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int i = q >> 3, c = (q >> 1) & 3, j = q & 1;
      meetings[(grp * 16 + q) * 64 + lane] = v4f{acc[i][j][4 * c], acc[i][j][4 * c + 1], acc[i][j][4 * c + 2], acc[i][j][4 * c + 3]};
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < QPW; ++q) {
      sum[q] = meetings[(grp * QPW + q) * 64 + lane];
#pragma unroll
      for (int o = 1; o < KG; ++o) {
        const v4f w = meetings[(o * 16 + grp * QPW + q) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[q][e] += w[e];
      }
    }
  };
  v4f sum[QPW];
  meet(sum);
  const unsigned ldc = p.ldc, col = n0 + 2 * lrow;
  auto rowOf = [&](int x, int e) {  // of quads 2 x and 2 x + 1
    const int q = grp * QPW + 2 * x;
    return m0 + 32 * (q >> 3) + 8 * ((q >> 1) & 3) + 4 * g + e;
  };
  float notFinite = 0.f, low = 1.f;
#pragma unroll
  for (int x = 0; x < QPW / 2; ++x)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        notFinite = fmaf(sum[2 * x + j][e], 0.f, notFinite);
        low = rowOf(x, e) < M && col + j < N ? fminf(low, __builtin_fabsf(sum[2 * x + j][e])) : low;
      }
  constexpr int MINE = QPW / 4;  // the thread's results, in sixteens
  auto value = [&](auto block, auto r) __attribute__((always_inline)) -> float {
    const float v = sum[4 * block + r / 4][(int)(r % 4)];  // (a copy: a bit_cast of a vector's element reads its first one)
    return v;
  };
  auto where = [&](int block, int r, unsigned& row, unsigned& column) __attribute__((always_inline)) {
    row = rowOf((4 * block + r / 4) / 2, r % 4) - m0;
    column = 2 * lrow + (r / 4) % 2;
  };
  unsigned again[MINE];
  auto raise = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i)  // (a load of four columns that N cuts holds values of the next row: no columns of the matrix)
      if (i < 2 || col + i - 2 < N)
        __hip_atomic_fetch_max(&found.largest[i < 2 ? 32 * i + lrow : BM + 2 * lrow + i - 2], __builtin_bit_cast(unsigned, largest[i]),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  const bool suspicious = notFinite != 0.f || low < 0x1p-64f || fmaxf(fmaxf(largest[0], largest[1]), fmaxf(largest[2], largest[3])) >= 0x1p30f;
  if (split_failed<BM, BN, 64 * KG, TRANSB, MINE>(p, tile, suspicious, found, again, value, where, raise)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = v16f{};
    for (unsigned s = 0; s < steps; ++s) {
      float x[8][2], y[8][2];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const unsigned kk = firstK(s) + 2 * e + g;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const unsigned row = m0 + 32 * i + lrow, c = col + i;
          x[e][i] = kk < K && row < M ? tile.A[(size_t)row * lda + kk] : 0.f;
          y[e][i] = kk < K && c < N ? TRANSB ? tile.B[(size_t)c * ldb + kk] : tile.B[(size_t)kk * ldb + c] : 0.f;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e][i], y[e][j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
    v4f exact[QPW];
    meet(exact);
#pragma unroll
    for (int q = 0; q < QPW; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[q][e] = again[q / 4] >> (4 * (q % 4) + e) & 1 ? exact[q][e] : sum[q][e];
  }

  // ---- tile store: + bias, + residual, GELU
  float bv[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) bv[j] = tile.bias && col + j < N ? tile.bias[col + j] : 0.f;
#pragma unroll
  for (int x = 0; x < QPW / 2; ++x)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned row = rowOf(x, e);
      if (row >= M) continue;
      float v[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        v[j] = sum[2 * x + j][e] + bv[j];
        if (tile.R && col + j < N) v[j] += tile.R[(size_t)row * N + col + j];
        // same expression as the stand-alone GELU kernel, so that fusing changes no bit
        if (p.act == 1) v[j] = gelu_erf_f32(v[j]);
      }
      float* to = tile.C + (size_t)row * ldc + col;
      if (col + 1 < N && ((uintptr_t)to & 7) == 0) *reinterpret_cast<v2f*>(to) = v2f{v[0], v[1]};
      else
#pragma unroll
        for (int j = 0; j < 2; ++j)
          if (col + j < N) to[j] = v[j];
    }
}

template <class Kernel>
int launch(hipStream_t stream, SgemmParams& p, Kernel kern, bool (&attrSet)[16], int bm, int bn, int threads, size_t lds) {
  if (!sgemm_detail::set_tiles(p, bm, bn)) return set_error(TFCC_ROCM_INVALID_ARGUMENT, "sgemm: too many tiles");
  int dev = 0;
  TFCC_HIP_CHECK(hipGetDevice(&dev));
  TFCC_REQUIRE(dev >= 0 && dev < 16, "device index %d", dev);
  if (!attrSet[dev]) {  // per device: the attribute belongs to the function on one device
    TFCC_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attrSet[dev] = true;
  }
  hipLaunchKernelGGL(kern, dim3(p.chunk * 8), dim3(threads), lds, stream, p);
  return check_launch("sgemm");
}

template <int MI, int NI, int WGM, int WGN, int KG, bool TRANSB>
int launch_shared(hipStream_t stream, SgemmParams p) {
  constexpr int BM = 32 * MI * WGM, BN = 32 * NI * WGN;
  constexpr size_t lds = KG * 3 * SharedLayout<BM, BN>::STAGE;
  static_assert(lds <= 159 * 1024, "LDS budget");
  static bool attrSet[16] = {};
  return launch(stream, p, sgemm_split_kernel<MI, NI, WGM, WGN, KG, TRANSB>, attrSet, BM, BN, 64 * WGM * WGN * KG, lds);
}

template <int KG, bool TRANSB>
int launch64(hipStream_t stream, SgemmParams p) {
  static bool attrSet[16] = {};
  return launch(stream, p, sgemm_split64_kernel<KG, TRANSB>, attrSet, 64, 64, 64 * KG, (size_t)KG * 64 * 64 * 4);
}

}  // namespace

namespace sgemm_detail {

int sgemm_split_launch(hipStream_t stream, const SgemmParams& p, int kernel, bool transB) {
  switch (kernel) {
    case sgemm_split_plan::kWide: return transB ? launch_shared<2, 2, 2, 4, 1, true>(stream, p) : launch_shared<2, 2, 2, 4, 1, false>(stream, p);
    case sgemm_split_plan::k128: {
      // (of one product: one of a group is summed as it is alone)
      const unsigned long long tiles = sgemm_tiles::tiles_of(p.M, p.N, p.groups ? 1 : p.batch, 128, 128);
      if (sgemm_split_plan::k_groups_of_128(tiles, p.K) == 2)
        return transB ? launch_shared<2, 2, 2, 2, 2, true>(stream, p) : launch_shared<2, 2, 2, 2, 2, false>(stream, p);
      return transB ? launch_shared<2, 2, 2, 2, 1, true>(stream, p) : launch_shared<2, 2, 2, 2, 1, false>(stream, p);
    }
    default: return transB ? launch64<4, true>(stream, p) : launch64<4, false>(stream, p);
  }
}

}  // namespace sgemm_detail
}  // namespace tfcc_rocm
