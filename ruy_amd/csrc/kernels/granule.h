// Reading rows of any alignment and length 16 bytes at a time.
#ifndef RUY_AMD_CSRC_KERNELS_GRANULE_H_
#define RUY_AMD_CSRC_KERNELS_GRANULE_H_

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ruyamd {
namespace granule {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef v4i v4i_unaligned __attribute__((aligned(1)));

// Low `n` bytes of a 32-bit word (n <= 0: none, n >= 4: all).
__device__ __forceinline__ uint32_t LowBytes(int n) {
  return n >= 4 ? 0xffffffffu : n <= 0 ? 0u : (1u << (8 * n)) - 1u;
}

// The granule (16 bytes) at depth byte k of a row of `bytes` bytes (kShort: less
// than 16), without reading outside the row. Global memory takes any byte
// address, so that is one load; a granule that reaches past the row's end is
// taken from the 16 bytes that end there and moved down to where it belongs
// afterwards, zeros following. Load and rest are apart so that a lane's loads
// are all issued before the first is waited for.
// An address that is no multiple of 4 costs a CU's address unit four times the
// cycles of an aligned one. That does not show where a kernel waits for memory,
// as the pack does (8192 rows of 8177 bytes 22.6 us at a pitch of 8192, 22.4 at
// 8179; 2048 of 4097 7.5 at 4112, 7.9 at 4099), but it does where a CU reads
// rows from its cache as fast as it can (mfma_gemm.h, kStagedBytes).
template <bool kShort>
__device__ __forceinline__ v4i LoadGranule(const uint8_t* row, int k, int bytes) {
  if constexpr (!kShort) return *reinterpret_cast<const v4i_unaligned*>(row + min(k, bytes - 16));
  v4i x = {0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < 15; ++i)
    if (i < bytes) x[i / 4] |= static_cast<int>(uint32_t(row[i]) << (8 * (i & 3)));
  return x;
}
template <bool kShort = false>
__device__ __forceinline__ v4i PlaceGranule(v4i x, int k, int bytes) {
  if constexpr (kShort) return k == 0 ? x : v4i{0, 0, 0, 0};
  const int shift = k - min(k, bytes - 16);  // 0: a whole granule; 16 and more: nothing of the row
  if (shift & 8) x = v4i{x[2], x[3], 0, 0};
  if (shift & 4) x = v4i{x[1], x[2], x[3], 0};
  const int s = shift & 3;
  x[0] = static_cast<int>(__builtin_amdgcn_alignbyte(x[1], x[0], s));
  x[1] = static_cast<int>(__builtin_amdgcn_alignbyte(x[2], x[1], s));
  x[2] = static_cast<int>(__builtin_amdgcn_alignbyte(x[3], x[2], s));
  x[3] = static_cast<int>(__builtin_amdgcn_alignbyte(0, x[3], s));
  if (k >= bytes) x = v4i{0, 0, 0, 0};
  return x;
}

}  // namespace granule
}  // namespace ruyamd

#endif  // RUY_AMD_CSRC_KERNELS_GRANULE_H_
