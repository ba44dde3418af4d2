// Moves between device memory and page-locked host memory as kernels on the caller's stream.  A copy engine command
// costs about 10 us before its first byte and another wait behind it; a launch costs 3 us, and its last workgroup can
// tell the waiting host itself.
#include "common.hpp"

namespace tfcc_rocm {
namespace {

constexpr unsigned kMaxPieces = 16;      // descriptors that travel in the argument block

struct Pieces {
  const char* src[kMaxPieces];
  char* dst[kMaxPieces];
  unsigned long long bytes[kMaxPieces];
  unsigned firstBlock[kMaxPieces];
  unsigned count;
};

// Bytes of one workgroup: 256 lanes, QUADS 16-byte pieces each.  Small transfers are bound by the trip over PCIe and by how
// many workgroups ask at once, large ones by PCIe, where fewer workgroups with more under way each are faster.  us with
// 4 KB and with 16 KB, in order on a stream: in, 16 KB 2.9 and 7.2, 87 KB 4.3 and 7.9, 256 KB 8.0 and 8.8, 512 KB 14.5 and
// 13.2, 3 MB 76 and 60; out, 87 KB 4.1 and 5.6, 512 KB 11.8 and 13.9, 1 MB 21.8 and 22.9, 3 MB 64.6 and 60.5.
constexpr unsigned block_bytes(int quads) { return 256u * 16u * quads; }
constexpr size_t kManyBlocksIn = 384 * 1024, kManyBlocksOut = 1536 * 1024;  // bytes of a launch up to which a workgroup takes 4 KB

typedef unsigned transfer_v4u __attribute__((ext_vector_type(4)));
constexpr int kSystemScope = 1 | 16;  // sc0 sc1: the store goes through all caches

// Workgroup `block` of the piece: its QUADS 4 KB.  All loads are asked for before the first store, so that a lane has
// 16 QUADS bytes under way on PCIe.  TO_HOST: the stores are done, for the host as well, when they are counted as such.
template <int QUADS, bool TO_HOST>
__device__ __forceinline__ void copy_block(const char* __restrict__ src, char* __restrict__ dst, unsigned long long bytes,
                                           unsigned block) {
  const unsigned long long begin = (unsigned long long)block * block_bytes(QUADS);
  const unsigned long long left = bytes - begin;
  const unsigned n = left < block_bytes(QUADS) ? (unsigned)left : block_bytes(QUADS);
  src += begin;
  dst += begin;
  auto byte = [&](unsigned i) {
    if constexpr (TO_HOST) __hip_atomic_store(dst + i, src[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else dst[i] = src[i];
  };
  if (((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15u) == 0) {
    const unsigned whole = n / 16;
    const transfer_v4u* s = reinterpret_cast<const transfer_v4u*>(src);
    const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc(dst, 0, (int)n, 0x00020000);
    transfer_v4u v[QUADS];
#pragma unroll
    for (unsigned q = 0; q < QUADS; ++q)
      if (q * 256 + threadIdx.x < whole) v[q] = s[q * 256 + threadIdx.x];
#pragma unroll
    for (unsigned q = 0; q < QUADS; ++q)
      if (q * 256 + threadIdx.x < whole)
        __builtin_amdgcn_raw_buffer_store_b128(v[q], d, (q * 256 + threadIdx.x) * 16u, 0, TO_HOST ? kSystemScope : 0);
    for (unsigned i = whole * 16 + threadIdx.x; i < n; i += 256) byte(i);
  } else {
    for (unsigned i = threadIdx.x; i < n; i += 256) byte(i);
  }
}

template <int QUADS, bool TO_HOST>
__device__ __forceinline__ void copy_pieces(const Pieces& p) {
  unsigned i = 0;
  while (i + 1 < p.count && blockIdx.x >= p.firstBlock[i + 1]) ++i;
  copy_block<QUADS, TO_HOST>(p.src[i], p.dst[i], p.bytes[i], blockIdx.x - p.firstBlock[i]);
}

template <int QUADS>
__global__ __launch_bounds__(256) void scatter_kernel(Pieces p) {
  copy_pieces<QUADS, false>(p);
}

// Bound by PCIe (57 GB/s): 3 MB in 60 us.  The last workgroup to arrive raises *flag to `epoch`, which the host polls:
// it sees a 4 KB result 6.8 us after the launch call, where waiting for the stream takes 11.7 us.  The results go through
// all caches by themselves, so waiting for them is all the order there has to be (with a fence for the whole system in every
// workgroup, which writes back what the kernels before have left in the L2s, 3 MB 72 us, 87 KB 6.9 instead of 4.1).
template <int QUADS>
__global__ __launch_bounds__(256) void gather_kernel(Pieces p, unsigned* arrivals, unsigned* flag, unsigned epoch) {
  copy_pieces<QUADS, true>(p);
  if (flag == nullptr) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wavefront's own stores are in host memory before the barrier lets it go
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned before = __hip_atomic_fetch_add(arrivals, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (before + 1 == gridDim.x) {
      __hip_atomic_store(arrivals, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the stream's next launch
      __hip_atomic_store(flag, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// launch(pieces, workgroups, whether they take 4 KB each, whether it is the last one), kMaxPieces at a time
template <class Launch>
int launch_pieces(const char* what, const tfcc_rocm_copy_piece* pieces, unsigned count, size_t manyBlocks, Launch&& launch) {
  for (unsigned i = 0; i < count; ++i)
    TFCC_REQUIRE(pieces[i].src && pieces[i].dst && pieces[i].bytes > 0 && pieces[i].bytes <= (1ull << 40), "%s: bad piece %u", what, i);
  for (unsigned at = 0; at < count; at += kMaxPieces) {
    Pieces p;
    p.count = count - at < kMaxPieces ? count - at : kMaxPieces;
    unsigned long long blocks = 0, bytes = 0;
    for (unsigned i = 0; i < p.count; ++i) bytes += pieces[at + i].bytes;
    const bool many = bytes <= manyBlocks;
    const unsigned each = block_bytes(many ? 1 : 4);
    for (unsigned i = 0; i < p.count; ++i) {
      p.src[i] = static_cast<const char*>(pieces[at + i].src);
      p.dst[i] = static_cast<char*>(pieces[at + i].dst);
      p.bytes[i] = pieces[at + i].bytes;
      p.firstBlock[i] = (unsigned)blocks;
      blocks += (pieces[at + i].bytes + each - 1) / each;
      TFCC_REQUIRE(blocks <= 0x7fffffffu, "%s: too many bytes", what);
    }
    launch(p, (unsigned)blocks, many, at + kMaxPieces >= count);
    if (int e = check_launch(what)) return e;
  }
  return TFCC_ROCM_OK;
}

}  // namespace
}  // namespace tfcc_rocm

using namespace tfcc_rocm;

extern "C" {

int tfcc_rocm_host_malloc(void** ptr, size_t bytes) {
  TFCC_REQUIRE(ptr != nullptr, "host_malloc: null argument");
  *ptr = nullptr;
  TFCC_HIP_CHECK(hipHostMalloc(ptr, bytes, hipHostMallocPortable | hipHostMallocCoherent));
  return TFCC_ROCM_OK;
}

int tfcc_rocm_host_free(void* ptr) {
  if (ptr == nullptr) return TFCC_ROCM_OK;
  TFCC_HIP_CHECK(hipHostFree(ptr));
  return TFCC_ROCM_OK;
}

int tfcc_rocm_copy_from_pinned(void* stream, void* dst_device, const void* src_pinned, size_t bytes) {
  if (bytes == 0) return TFCC_ROCM_OK;
  TFCC_REQUIRE(dst_device && src_pinned, "copy_from_pinned: null argument");
  const tfcc_rocm_copy_piece piece = {src_pinned, dst_device, bytes};
  return tfcc_rocm_copy_pieces_from_pinned(stream, &piece, 1);
}

int tfcc_rocm_copy_pieces_from_pinned(void* stream, const tfcc_rocm_copy_piece* pieces, unsigned count) {
  TFCC_REQUIRE(pieces && count > 0, "copy_from_pinned: null argument");
  return launch_pieces("copy_from_pinned", pieces, count, kManyBlocksIn, [&](const Pieces& p, unsigned blocks, bool many, bool) {
    hipLaunchKernelGGL(many ? scatter_kernel<1> : scatter_kernel<4>, dim3(blocks), dim3(256), 0, as_stream(stream), p);
  });
}

int tfcc_rocm_copy_to_pinned(void* stream, const tfcc_rocm_copy_piece* pieces, unsigned count, unsigned* arrivals_device,
                             unsigned* flag_pinned, unsigned epoch) {
  TFCC_REQUIRE(pieces && count > 0 && arrivals_device && flag_pinned, "copy_to_pinned: null argument");
  // the stream runs the launches in order: only the last one tells the host
  return launch_pieces("copy_to_pinned", pieces, count, kManyBlocksOut, [&](const Pieces& p, unsigned blocks, bool many, bool last) {
    hipLaunchKernelGGL(many ? gather_kernel<1> : gather_kernel<4>, dim3(blocks), dim3(256), 0, as_stream(stream), p, arrivals_device,
                       last ? flag_pinned : nullptr, epoch);
  });
}

}  // extern "C"
