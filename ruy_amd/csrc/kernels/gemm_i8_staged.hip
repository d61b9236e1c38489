// The int8 GEMM on operands of any alignment and depth, read through registers
// instead of being packed first (mfma_gemm.h, kStaged).
#include <hip/hip_runtime.h>

#include "int8_traits.h"
#include "mfma_gemm.h"

namespace ruyamd {

// Where all workgroups run at once - two to a CU with the ring of four stages,
// one with that of eight - the product is little more than its launch, one
// round trip to memory and its write-back, and a pack launch in front costs two
// thirds of that again: 1024 x 333 x 1024 9.4 us packed, 6.6 staged; 1024 x
// 1023 x 1024 11.9 and 9.9 (8.4 at a depth of 1020, whose rows start at whole
// dwords), 4236 x 106 x 256 10.0 and 5.9, 64 x 147 x 12544 uint8 9.5 and 6.0.
// In rounds it loses to larger tiles on packed operands: 2048 x 251 x 2048
// (1024 tiles of 64x64) 11.1 packed and 11.7 staged, 1500 x 1000 x 1500 (576)
// 17.1 and 21.8.
// (What the 32x32 tiles take, PlanSmallGemmI8, never gets here.)
// Operands that can be used in place gain less, since nothing is packed (us per
// call, direct -> staged). Up to 384 bytes of depth the direct loads are as good
// on one workgroup a CU (256^3 4.8, staged 5.0), from 900 on the schedule that
// deals the depth to the waves; in between it wins (512^3 4.7 -> 4.3, 1024 x 640 x
// 1024 5.4 -> 4.8), but not with the end of a row that is no whole number of
// 128-byte stages, which costs it some 0.6 us more than a direct load of it (1024
// x 400 x 1024 4.9 -> 5.6, 1024 x 720 x 640 5.7 -> 6.8, with sums 753 x 720 x 640
// 7.1 -> 7.7: every one of 100 such shapes is slower staged).
// Where two workgroups a CU take a grid that would otherwise go to a larger tile
// it wins on whole stages (2048 x 128 x 1024 4.7 -> 4.3, with sums 6.1 -> 4.8,
// 4096 x 256 x 512 with sums 7.0 -> 5.6, 2048 x 512 x 1024 with sums 7.0 -> 6.7,
// without: even) and where it forms sums as well, for which other tiles need a
// round of their own (1300 x 176 x 1300 7.2 -> 6.5, 2040 x 368 x 801 8.5 -> 7.1,
// 4088 x 448 x 417 8.6 -> 7.7, 2048 x 272 x 929 even). A part of a stage without
// sums is the larger tile's (2048 x 320 x 1024 5.4, staged 6.0, 1249 x 496 x 801
// 6.4 and 7.1) while less than half a run of 16 rows is left over at the end of a
// column, which it stores one by one with twice the blocks to a wave: of 90
// shapes 3 to 14 % faster up to 5 such rows, 8 faster to 3 slower at 6 and 7, from
// 8 on 3 faster to 6 slower (2043 x 368 x 896 7.2 -> 6.8, 1416 x 144 x 705 6.4 -> 6.1).
bool GemmI8StagedIsBetter(const GemmArgs& args, int num_cus, int depth, bool in_place) {
  if (depth < 16 || depth > kGemmI8StagedDepth) return false;
  if (args.forced_tile_rows && (in_place || args.forced_tile_rows != 64 || args.forced_tile_cols != 64)) return false;
  const int tiles = mfma_gemm::TileCount(args, 64, 64);
  if (tiles > num_cus * (depth <= 512 ? 2 : 1)) return false;
  if (!in_place) return true;
  if (tiles > num_cus) return depth % 128 == 0 || args.fuse_sums || args.M % 16 >= 8;
  return depth % 128 == 0 && depth > 384 && depth <= 896;
}

namespace {

template <int kStages, int kForm>
hipError_t LaunchForm(hipStream_t stream, const GemmArgs& args) {
  return args.fuse_sums
             ? mfma_gemm::Launch<Int8Traits, 1, 1, 128, kStages, true, false, false, false, false, kForm>(stream, args)
             : mfma_gemm::Launch<Int8Traits, 1, 1, 128, kStages, false, false, false, false, false, kForm>(stream, args);
}

}  // namespace

hipError_t LaunchGemmI8Staged(hipStream_t stream, const GemmArgs& args) {
  if (args.k_valid < 16 || args.k_valid > kGemmI8StagedDepth || args.k_bytes != (args.k_valid + 15) / 16 * 16 ||
      args.row_sums || args.split_k != 1)
    return hipErrorInvalidValue;
  const bool dwords = ((reinterpret_cast<uintptr_t>(args.a) | reinterpret_cast<uintptr_t>(args.b) |
                        static_cast<uint32_t>(args.lda) | static_cast<uint32_t>(args.ldb)) & 3) == 0;
  if (args.k_valid <= 512) {
    return dwords ? LaunchForm<4, mfma_gemm::kStagedDwords>(stream, args)
                  : LaunchForm<4, mfma_gemm::kStagedBytes>(stream, args);
  }
  return dwords ? LaunchForm<8, mfma_gemm::kStagedDwords>(stream, args)
                : LaunchForm<8, mfma_gemm::kStagedBytes>(stream, args);
}

}  // namespace ruyamd
