// Small transfers between page-locked host memory and the device for callers
// that hand over host pointers. A call that stages its operands through the
// copy engines pays for more than the bytes: every transfer goes through the
// queue of another engine, whose start waits for a signal of the one before
// and whose end the kernel behind it waits for in turn, and the host learns of
// the last one through an event. Up to some hundreds of KiB that is all of the
// time (1024 x 1024 x 196 int8 with cached weights, 200 KB each way: 73 to
// 106 us per call, of which the product takes 7 us and the bytes 4 us a
// direction; 40 us this way).
// Here everything a call uploads goes in one launch on the call's own stream,
// the result comes back by another, and the host reads its completion from
// words that the second one leaves in host memory.
#include "host_copy.h"

namespace ruyamd {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kPerThread = int(kHostCopyBlockBytes) / 16 / kThreads;

// 16 KiB per workgroup, four 16-byte accesses per thread: bound by PCIe and its
// latency. kTogether: a thread's four loads are in flight together, those past the
// end reading the last granule; otherwise each stands behind a bounds test of its
// own and is awaited there, which is what large uploads want (LaunchUpload).
// Downloads, which load from device memory, always gain by it: whole calls 0.3 to 1
// us (1024 x 1024 x 196 with cached weights 37.7 -> 37.2, 512 KiB down 47.6 -> 47.5).
template <bool kTogether>
__device__ __forceinline__ void CopyBlock(const void* from, void* to, uint32_t bytes) {
  const int granules = static_cast<int>((bytes + 15) / 16);
  const int first = int(blockIdx.x) * kThreads * kPerThread + int(threadIdx.x);
  const v4i* s = static_cast<const v4i*>(from);
  v4i* d = static_cast<v4i*>(to);
  v4i x[kPerThread];
#pragma unroll
  for (int i = 0; i < kPerThread; ++i) {
    if constexpr (kTogether)
      x[i] = s[min(first + i * kThreads, granules - 1)];
    else if (first + i * kThreads < granules)
      x[i] = s[first + i * kThreads];
  }
#pragma unroll
  for (int i = 0; i < kPerThread; ++i)
    if (first + i * kThreads < granules) d[first + i * kThreads] = x[i];
}

template <bool kTogether>
__global__ __launch_bounds__(kThreads) void UploadKernel(UploadPieces pieces) {
  const uint32_t bytes = pieces.bytes[blockIdx.y];
  // (A launch has as many workgroups to a piece as the longest needs.)
  if (blockIdx.x * uint32_t(kHostCopyBlockBytes) >= bytes) return;
  CopyBlock<kTogether>(pieces.from[blockIdx.y], pieces.to[blockIdx.y], bytes);
}

__global__ __launch_bounds__(kThreads) void DownloadKernel(const void* from, void* to, uint32_t bytes, uint32_t* done,
                                                           uint32_t value) {
  CopyBlock<true>(from, to, bytes);
  // Every wave writes back and awaits its own stores before the barrier: the
  // barrier itself waits for no store, and the release behind it only for those
  // of the one wave that stores the word.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(done + blockIdx.x, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

hipError_t LaunchUpload(hipStream_t stream, const UploadPieces& pieces) {
  uint32_t most = 0;
  uint64_t all = 0;
  for (int i = 0; i < pieces.count; ++i) {
    most = pieces.bytes[i] > most ? pieces.bytes[i] : most;
    all += pieces.bytes[i];
  }
  if (most == 0) return hipSuccess;
  const unsigned blocks = static_cast<unsigned>((most + kHostCopyBlockBytes - 1) / kHostCopyBlockBytes);
  // More reads than this outstanding over PCIe only get in each other's way. Whole
  // calls, one after the other -> together: 50 KiB up 25.0 -> 21.5 us, 128 28.7 -> 26.1,
  // 196 37.7 -> 36.2, 320 41.8 -> 41.7, 512 48.3 -> 49.0, 780 91.8 -> 92.5, 2048 148 -> 158.
  constexpr uint64_t kMostTogether = 256 * 1024;
  const bool together = all <= kMostTogether;
  hipLaunchKernelGGL(together ? UploadKernel<true> : UploadKernel<false>, dim3(blocks, pieces.count), dim3(kThreads), 0,
                     stream, pieces);
  return hipGetLastError();
}

hipError_t LaunchDownload(hipStream_t stream, const void* from, void* to, std::size_t bytes, uint32_t* done,
                          uint32_t value) {
  if (bytes == 0) return hipSuccess;
  hipLaunchKernelGGL(DownloadKernel, dim3(DownloadBlocks(bytes)), dim3(kThreads), 0, stream, from, to,
                     static_cast<uint32_t>(bytes), done, value);
  return hipGetLastError();
}

}  // namespace ruyamd
