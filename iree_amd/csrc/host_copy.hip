// Copies between the host's pinned memory and the device, as kernels on the
// caller's stream (uk_api.hip mirrors host operands with them).
//
// The copy engines move large pieces at the same rate (50 to 55 GB/s each way),
// but work that goes from an engine to a kernel and back waits for the hand-over
// each time: 80 KB up, a product and 64 KB down take 35 us with engine copies and
// 20 us with these, in one queue with the product.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "uk_internal.h"

namespace uk {
namespace {

typedef int v4i32 __attribute__((ext_vector_type(4)));

struct UploadArgs {
  const v4i32* src;  // pinned
  v4i32* dst;
  int32_t vecs;
};

// 64 workgroups with four loads per lane in flight: more of either moves less (52.6 GB/s at 8 MiB, 44 with 1024
// workgroups).
__global__ __launch_bounds__(256) void upload_kernel(const UploadArgs a) {
  const int stride = gridDim.x * 256;
  int i = blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * stride < a.vecs; i += 4 * stride) {
    v4i32 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = a.src[i + u * stride];
#pragma unroll
    for (int u = 0; u < 4; ++u) a.dst[i + u * stride] = v[u];
  }
  for (; i < a.vecs; i += stride) a.dst[i] = a.src[i];
}

struct DownloadArgs {
  const v4i32* src;
  v4i32* dst;       // pinned
  uint32_t* flags;  // pinned, one per piece
  uint32_t generation;
  int32_t vecs, pieces;
};

// Workgroups copy pieces in order and then set their flags to `generation`: the host takes the pieces as they arrive.
// (kDownloadGroups workgroups only: with one per piece all of them would arrive at the end.)
constexpr int kDownloadGroups = 16;
__global__ __launch_bounds__(256) void download_kernel(const DownloadArgs a) {
  constexpr int PER_LANE = kDownloadPieceBytes / 16 / 256;
  for (int piece = blockIdx.x; piece < a.pieces; piece += kDownloadGroups) {
    const int first = piece * (kDownloadPieceBytes / 16) + threadIdx.x;
    v4i32 v[PER_LANE];
#pragma unroll
    for (int u = 0; u < PER_LANE; ++u)
      if (first + 256 * u < a.vecs) v[u] = a.src[first + 256 * u];
#pragma unroll
    for (int u = 0; u < PER_LANE; ++u)
      if (first + 256 * u < a.vecs) a.dst[first + 256 * u] = v[u];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(a.flags + piece, a.generation, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace

hipError_t launch_upload(const void* pinned, void* dst, size_t bytes, hipStream_t stream) {
  UploadArgs a{(const v4i32*)pinned, (v4i32*)dst, (int32_t)((bytes + 15) / 16)};
  const unsigned blocks = (unsigned)((a.vecs + 255) / 256);
  return launch_kernel(upload_kernel, blocks < 64 ? blocks : 64, 256, 0, stream, a);
}

hipError_t launch_download(const void* src, void* pinned, uint32_t* flags, uint32_t generation, size_t bytes,
                           hipStream_t stream) {
  const int32_t pieces = (int32_t)((bytes + kDownloadPieceBytes - 1) / kDownloadPieceBytes);
  DownloadArgs a{(const v4i32*)src, (v4i32*)pinned, flags, generation, (int32_t)((bytes + 15) / 16), pieces};
  return launch_kernel(download_kernel, pieces < kDownloadGroups ? pieces : kDownloadGroups, 256, 0, stream, a);
}

}  // namespace uk
