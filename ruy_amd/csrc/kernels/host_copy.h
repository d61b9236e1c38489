// Copies between page-locked host memory and device memory by kernels.
#ifndef RUY_AMD_CSRC_KERNELS_HOST_COPY_H_
#define RUY_AMD_CSRC_KERNELS_HOST_COPY_H_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace ruyamd {

// What one launch moves to the device: up to kMost pieces of page-locked host
// memory. Both addresses are multiples of 16; `bytes` is rounded up to 16 when
// copying, so both sides must have that much room.
struct UploadPieces {
  static constexpr int kMost = 8;
  int count = 0;
  const void* from[kMost] = {};
  void* to[kMost] = {};
  uint32_t bytes[kMost] = {};
};
hipError_t LaunchUpload(hipStream_t stream, const UploadPieces& pieces);

// Bytes a workgroup of the two kernels copies.
constexpr std::size_t kHostCopyBlockBytes = 16384;
inline int DownloadBlocks(std::size_t bytes) {
  return static_cast<int>((bytes + kHostCopyBlockBytes - 1) / kHostCopyBlockBytes);
}

// to[0, bytes) = from[0, bytes) with `to` and `done` in page-locked, coherent
// host memory; workgroup b then stores `value` to done[b] (DownloadBlocks(bytes)
// words), so that a host that reads `value` in every word finds the copy
// complete. Addresses and rounding as above.
hipError_t LaunchDownload(hipStream_t stream, const void* from, void* to, std::size_t bytes, uint32_t* done,
                          uint32_t value);

}  // namespace ruyamd

#endif  // RUY_AMD_CSRC_KERNELS_HOST_COPY_H_
