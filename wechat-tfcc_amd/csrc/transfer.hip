// Moves between device memory and page-locked host memory as kernels on the caller's stream.  A copy engine command
// costs about 10 us before its first byte and another wait behind it; a launch costs 3 us, and its last workgroup can
// tell the waiting host itself.
#include "common.hpp"

namespace tfcc_rocm {
namespace {

constexpr unsigned kBlockBytes = 16384;  // of one workgroup: 256 lanes, four 16-byte pieces each
constexpr unsigned kMaxPieces = 16;      // descriptors that travel in the argument block

struct Pieces {
  const char* src[kMaxPieces];
  char* dst[kMaxPieces];
  unsigned long long bytes[kMaxPieces];
  unsigned firstBlock[kMaxPieces];
  unsigned count;
};

// Workgroup `block` of the piece: bytes [block * 16 KB, + 16 KB) of it.  All four loads are asked for before the first
// store, so that a lane has 64 bytes under way on PCIe.
__device__ __forceinline__ void copy_block(const char* __restrict__ src, char* __restrict__ dst, unsigned long long bytes,
                                           unsigned block) {
  const unsigned long long begin = (unsigned long long)block * kBlockBytes;
  const unsigned long long left = bytes - begin;
  const unsigned n = left < kBlockBytes ? (unsigned)left : kBlockBytes;
  src += begin;
  dst += begin;
  if (((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15u) == 0) {
    const unsigned whole = n / 16;
    const uint4* s = reinterpret_cast<const uint4*>(src);
    uint4* d = reinterpret_cast<uint4*>(dst);
    uint4 v[4];
#pragma unroll
    for (unsigned q = 0; q < 4; ++q)
      if (q * 256 + threadIdx.x < whole) v[q] = s[q * 256 + threadIdx.x];
#pragma unroll
    for (unsigned q = 0; q < 4; ++q)
      if (q * 256 + threadIdx.x < whole) d[q * 256 + threadIdx.x] = v[q];
    for (unsigned i = whole * 16 + threadIdx.x; i < n; i += 256) dst[i] = src[i];
  } else {
    for (unsigned i = threadIdx.x; i < n; i += 256) dst[i] = src[i];
  }
}

__global__ __launch_bounds__(256) void copy_kernel(const char* src, char* dst, unsigned long long bytes) {
  copy_block(src, dst, bytes, blockIdx.x);
}

// Bound by PCIe (57 GB/s): 3 MB in 62 us.  The last workgroup to arrive raises *flag to `epoch`, which the host polls:
// it sees a 4 KB result 7.4 us after the launch call, where waiting for the stream takes 11.7 us.
__global__ __launch_bounds__(256) void gather_kernel(Pieces p, unsigned* arrivals, unsigned* flag, unsigned epoch) {
  unsigned i = 0;
  while (i + 1 < p.count && blockIdx.x >= p.firstBlock[i + 1]) ++i;
  copy_block(p.src[i], p.dst[i], p.bytes[i], blockIdx.x - p.firstBlock[i]);
  if (flag == nullptr) return;
  __threadfence_system();  // every wavefront's own stores have reached host memory before the barrier lets it go
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned before = __hip_atomic_fetch_add(arrivals, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_SYSTEM);
    if (before + 1 == gridDim.x) {
      __hip_atomic_store(arrivals, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the stream's next launch
      __hip_atomic_store(flag, epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
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
  const size_t blocks = (bytes + kBlockBytes - 1) / kBlockBytes;
  TFCC_REQUIRE(blocks <= 0x7fffffffu, "copy_from_pinned: %zu bytes", bytes);
  hipLaunchKernelGGL(copy_kernel, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream),
                     static_cast<const char*>(src_pinned), static_cast<char*>(dst_device), (unsigned long long)bytes);
  return check_launch("copy_from_pinned");
}

int tfcc_rocm_copy_to_pinned(void* stream, const tfcc_rocm_copy_piece* pieces, unsigned count, unsigned* arrivals_device,
                             unsigned* flag_pinned, unsigned epoch) {
  TFCC_REQUIRE(pieces && count > 0 && arrivals_device && flag_pinned, "copy_to_pinned: null argument");
  for (unsigned i = 0; i < count; ++i)
    TFCC_REQUIRE(pieces[i].src && pieces[i].dst && pieces[i].bytes > 0 && pieces[i].bytes <= (1ull << 40),
                 "copy_to_pinned: bad piece %u", i);
  for (unsigned at = 0; at < count; at += kMaxPieces) {
    Pieces p;
    p.count = count - at < kMaxPieces ? count - at : kMaxPieces;
    unsigned long long blocks = 0;
    for (unsigned i = 0; i < p.count; ++i) {
      p.src[i] = static_cast<const char*>(pieces[at + i].src);
      p.dst[i] = static_cast<char*>(pieces[at + i].dst);
      p.bytes[i] = pieces[at + i].bytes;
      p.firstBlock[i] = (unsigned)blocks;
      blocks += (pieces[at + i].bytes + kBlockBytes - 1) / kBlockBytes;
      TFCC_REQUIRE(blocks <= 0x7fffffffu, "copy_to_pinned: too many bytes");
    }
    // the stream runs the launches in order: only the last one tells the host
    const bool last = at + kMaxPieces >= count;
    hipLaunchKernelGGL(gather_kernel, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream), p, arrivals_device,
                       last ? flag_pinned : nullptr, epoch);
    if (int e = check_launch("copy_to_pinned")) return e;
  }
  return TFCC_ROCM_OK;
}

}  // extern "C"
