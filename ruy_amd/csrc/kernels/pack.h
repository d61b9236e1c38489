// Launch interface of the pack kernels.
#ifndef RUY_AMD_CSRC_KERNELS_PACK_H_
#define RUY_AMD_CSRC_KERNELS_PACK_H_

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ruyamd {

// A matrix seen as `count` depth-vectors of length K: vector c, depth k is
// data[c * stride_c + k * stride_k] (elements of `dtype`). One of the two
// strides is 1.
struct PackSource {
  const void* data = nullptr;
  int64_t stride_c = 0;
  int64_t stride_k = 0;
  int32_t count = 0;
  int32_t K = 0;
  int32_t dtype = 0;
};

// One operand of an 8-bit or fp32 product to be re-laid out. The device form
// of the reference's Pack (ruy/pack.h:105-132 with the uint8 -> int8 conversion
// of ruy/pack_common.h:36-58): vector c goes to dst + c * ld (`ld` in bytes, a
// multiple of 16; 8-bit values as int8), zero-filled from its K values up to
// the end of their last 16 bytes. With `sums`, sums[c] becomes the sum of the packed 8-bit values; only for
// operands of which PackFormsSums says so.
struct PackJob {
  PackSource src;
  void* dst = nullptr;
  int32_t ld = 0;
  int32_t* sums = nullptr;
};
// Up to two of them (the two operands of a product) in one launch.
hipError_t LaunchPack(hipStream_t stream, const PackJob* jobs, int count);
// Whether the launch walks the whole depth of every vector in one place, so
// that the sums come with it. Otherwise whoever reads the packed operand forms
// them, like those of an operand used in place.
bool PackFormsSums(const PackSource& src);

// int16 operand for the int8 matrix cores: each value v is split into
// hi = v >> 8 (signed) and lo = (v & 0xff) - 128, both int8, so that
// v = 256*hi + lo + 128. For every group of 32 vectors the 32 hi vectors are
// written first, then the 32 lo vectors: vector c of plane p lands at
// dst + ((c/32)*64 + p*32 + c%32) * ld. Vectors past `count` inside the last
// group and depth past K are zero. The destination holds
// ceil(count/32)*64 vectors.
hipError_t LaunchPackI16Split(hipStream_t stream, const PackSource& src, int8_t* dst, int32_t ld);

}  // namespace ruyamd

#endif  // RUY_AMD_CSRC_KERNELS_PACK_H_
