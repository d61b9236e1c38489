// The int8 and int8 x int16 instantiations of the tiled matrix-core GEMM and
// the questions the planner asks about them.
#include <hip/hip_runtime.h>

#include <tuple>

#include "int8_traits.h"
#include "mfma_gemm.h"

namespace ruyamd {

bool GemmI8I16CanFuseSums(const GemmArgs& args, int num_cus) {
  return mfma_gemm::PickTile(args, num_cus, mfma_gemm::Model::kInt8PlaneSplit) == mfma_gemm::Tile::k64x128;
}

hipError_t LaunchGemmI8I16(hipStream_t stream, const GemmArgs& args, int num_cus) {
  if (args.fuse_sums) {
    if (!GemmI8I16CanFuseSums(args, num_cus)) return hipErrorInvalidValue;
    return mfma_gemm::LaunchSmallestTile<Int8SplitTraits, true>(stream, args);
  }
  return mfma_gemm::LaunchBest<Int8SplitTraits>(stream, args, num_cus);
}

bool GemmI8I16CanUseRawInt16(const GemmArgs& args, int num_cus) {
  if (!GemmI8I16CanFuseSums(args, num_cus)) return false;  // not the smallest tile
  const int k_tiles = (args.k_bytes + 127) / 128;
  const int parts = args.split_k > 1 ? args.split_k : 1;
  return (k_tiles + parts - 1) / parts >= 2;  // the schedule that deals the depth to the waves
}

hipError_t LaunchGemmI8I16Raw(hipStream_t stream, const GemmArgs& args, int num_cus) {
  if (!GemmI8I16CanUseRawInt16(args, num_cus)) return hipErrorInvalidValue;
  return args.fuse_sums ? mfma_gemm::Launch<Int8SplitRawTraits, 1, 2, 128, 4, true, false, true>(stream, args)
                        : mfma_gemm::Launch<Int8SplitRawTraits, 1, 2, 128, 4, false, false, true>(stream, args);
}

DepthSplit GemmDepthSplit(const GemmArgs& args, int num_cus, GemmKind kind) {
  const mfma_gemm::Model model = kind == GemmKind::kInt8Int16 ? mfma_gemm::Model::kInt8PlaneSplit
                                 : kind == GemmKind::kF32     ? mfma_gemm::Model::kF32
                                                              : mfma_gemm::Model::kInt8;
  return mfma_gemm::PlanDepthSplit(args, num_cus, model);
}

int GemmDepthSplitCounters() { return mfma_gemm::kSplitCounters; }

void GemmTileFor(const GemmArgs& args, int num_cus, GemmKind kind, int* tile_rows, int* tile_cols, int* depth_parts) {
  const mfma_gemm::Model which = kind == GemmKind::kInt8Int16 ? mfma_gemm::Model::kInt8PlaneSplit
                                 : kind == GemmKind::kF32     ? mfma_gemm::Model::kF32
                                                              : mfma_gemm::Model::kInt8;
  const DepthSplit split = mfma_gemm::PlanDepthSplit(args, num_cus, which);
  const mfma_gemm::Tile tile =
      split.large_tile ? mfma_gemm::Tile::k256x256 : mfma_gemm::ChooseTile(args, num_cus, which).tile;
  const mfma_gemm::TimingModel model = mfma_gemm::TimingModelOf(which);
  for (int i = 0; i < model.count; ++i) {
    if (model.tiles[i].tile == tile) {
      *tile_rows = model.tiles[i].bm;
      *tile_cols = model.tiles[i].bn;
    }
  }
  *depth_parts = split.parts;
}

bool GemmI8CanFuseSums(const GemmArgs& args, int num_cus) {
  const mfma_gemm::TileChoice choice = mfma_gemm::ChooseTile(args, num_cus, mfma_gemm::Model::kInt8);
  if (choice.large_parts != 1) return false;
  // (The smallest tile: unless sharing the rows out over its workgroups is cheaper.)
  if (choice.tile == mfma_gemm::Tile::k64x64) return !mfma_gemm::SmallestTileSharesSumsOut(args, num_cus);
  // The 128x128 tile forms the row sums of `a`, of `b` or of both, in grids
  // of at most one workgroup per CU.
  return choice.tile == mfma_gemm::Tile::k128x128 && mfma_gemm::RowSumming128Applies(args, num_cus);
}

// The smallest tile, asked after the depth split has been planned: the
// planner's answer, and every wave of the depth-per-wave schedule must have a
// step of the parts as they are.
static bool SmallestTileCanShareSumsOut(const GemmArgs& args, int num_cus) {
  if (args.split_large || !mfma_gemm::SmallestTileSharesSumsOut(args, num_cus)) return false;
  const int k_steps = std::max(1, (args.k_bytes + 127) / 128);
  const int parts = std::max(1, args.split_k);
  return parts <= k_steps && depth_split::StepsPerPart(k_steps, parts) >= 4 &&
         depth_split::NoEmptyPart(k_steps, parts);
}

bool GemmI8CanFormRowSums(const GemmArgs& args, int num_cus) {
  const bool flip = args.a_flip != 0 || args.b_flip != 0;
  const int tiles_m = (args.M + fused_sums::kTileRows - 1) / fused_sums::kTileRows;
  // (Asked after the depth split has been planned: every part needs its steps.)
  const int parts = args.split_k > 1 && args.split_large ? args.split_k : 1;
  const int steps = args.k_bytes / 128;
  // A row's sums take contributions from every part: the parts' workgroups
  // must all run at once, or the first ones wait (a bounded but long time) for
  // contributors that start when they are gone.
  const int tiles = tiles_m * ((args.N + fused_sums::kTileRows - 1) / fused_sums::kTileRows);
  if (parts > 1 && tiles * parts > num_cus) return false;
  // (uint8 data in place needs whole depth steps, which LaunchGemmI8 insists on.)
  if (flip && args.k_bytes % 128 != 0) return false;
  const mfma_gemm::Tile tile = mfma_gemm::PickTile(args, num_cus, mfma_gemm::Model::kInt8);
  if (tile == mfma_gemm::Tile::k64x64)
    return (args.sums_wanted & 1) && SmallestTileCanShareSumsOut(args, num_cus);
  // The tiles in between: by the workgroups of the grid, each for a share of the rows.
  for (const auto& [mid, bm, bn] : {std::tuple{mfma_gemm::Tile::k128x128, 128, 128},
                                    std::tuple{mfma_gemm::Tile::k128x64, 128, 64},
                                    std::tuple{mfma_gemm::Tile::k64x128, 64, 128}}) {
    if (tile == mid)
      return parts == 1 && mfma_gemm::LeadSumsApply(args, num_cus, bm, bn) &&
             mfma_gemm::LeadSumsMicroseconds(args, num_cus, bm, bn) <
                 mfma_gemm::SumsKernelMicroseconds(double(args.M) * args.k_bytes);
  }
  return depth_split::StepCount(steps, parts, parts - 1) >= fused_sums::kMinDepthSteps &&
         tiles_m * fused_sums::kTileRows <= fused_sums::kMaxRows && tile == mfma_gemm::Tile::k256x256;
}

bool GemmI8CanFormColumnSums(const GemmArgs& args, int num_cus, bool rows_in_launch) {
  if (args.split_k > 1 || !mfma_gemm::LeadColumnSumsApply(args)) return false;
  const bool flip = args.a_flip != 0 || args.b_flip != 0;
  if (flip && args.k_bytes % 128 != 0) return false;
  const mfma_gemm::Tile tile = mfma_gemm::PickTile(args, num_cus, mfma_gemm::Model::kInt8);
  if (tile == mfma_gemm::Tile::k64x64) return SmallestTileCanShareSumsOut(args, num_cus);
  // (The largest tile's kernel with sums in its launch always forms those of a's rows.)
  if (tile == mfma_gemm::Tile::k256x256 && !rows_in_launch) return false;
  for (const auto& [mid, bm, bn] : {std::tuple{mfma_gemm::Tile::k256x256, 256, 256},
                                    std::tuple{mfma_gemm::Tile::k128x128, 128, 128},
                                    std::tuple{mfma_gemm::Tile::k128x64, 128, 64},
                                    std::tuple{mfma_gemm::Tile::k64x128, 64, 128}}) {
    if (tile == mid)
      return mfma_gemm::LeadColumnSumsMicroseconds(args, num_cus, bm, bn) <
             mfma_gemm::SumsKernelMicroseconds(double(args.N) * args.k_bytes);
  }
  return false;
}

int GemmI8ColumnSumsOffset(const GemmArgs& args) { return mfma_gemm::ColumnSumsOffset(args); }

int GemmI8RowSumsProducers(const GemmArgs& args, int num_cus) {
  const mfma_gemm::Tile tile = mfma_gemm::PickTile(args, num_cus, mfma_gemm::Model::kInt8);
  if (tile == mfma_gemm::Tile::k128x128) return mfma_gemm::LeadSumsProducers(args, num_cus, 128, 128);
  if (tile == mfma_gemm::Tile::k128x64) return mfma_gemm::LeadSumsProducers(args, num_cus, 128, 64);
  if (tile == mfma_gemm::Tile::k64x128) return mfma_gemm::LeadSumsProducers(args, num_cus, 64, 128);
  if (tile == mfma_gemm::Tile::k256x256) return mfma_gemm::LeadSumsProducers(args, num_cus, 256, 256);
  if (tile == mfma_gemm::Tile::k64x64) return mfma_gemm::LeadSumsProducers(args, num_cus, 64, 64);
  return 0;
}

hipError_t LaunchGemmI8(hipStream_t stream, const GemmArgs& args, int num_cus) {
  const bool flip = args.a_flip != 0 || args.b_flip != 0;
  // Flipped bytes need a whole number of depth steps: bytes past the depth read as zero, which would turn into -128.
  if (flip && args.k_bytes % 128 != 0) return hipErrorInvalidValue;
  if (args.fuse_sums) {
    // Exists for the smallest tile and the 128x128 tile.
    if (!GemmI8CanFuseSums(args, num_cus)) return hipErrorInvalidValue;
    if (mfma_gemm::PickTile(args, num_cus, mfma_gemm::Model::kInt8) == mfma_gemm::Tile::k128x128 &&
        (args.sums_wanted & 2))
      return flip ? mfma_gemm::LaunchRowSumming128<Int8BothSums, true>(stream, args, num_cus)
                  : mfma_gemm::LaunchRowSumming128<Int8BothSums>(stream, args, num_cus);
    if (mfma_gemm::PickTile(args, num_cus, mfma_gemm::Model::kInt8) == mfma_gemm::Tile::k128x128)
      return flip ? mfma_gemm::LaunchRowSumming128<Int8Traits, true>(stream, args, num_cus)
                  : mfma_gemm::LaunchRowSumming128<Int8Traits>(stream, args, num_cus);
    return flip ? mfma_gemm::LaunchSmallestTile<Int8Traits, true, true>(stream, args)
                : mfma_gemm::LaunchSmallestTile<Int8Traits, true>(stream, args);
  }
  return flip ? mfma_gemm::LaunchBest<Int8Traits, true>(stream, args, num_cus)
              : mfma_gemm::LaunchBest<Int8Traits>(stream, args, num_cus);
}

hipError_t LaunchGemmI8Batch(hipStream_t stream, const GemmArgs& args, const GemmBatch& batch, int count,
                             int num_cus) {
  const bool flip = args.a_flip != 0 || args.b_flip != 0;
  // (Batches exist for the smallest tile.)
  if (mfma_gemm::PickTile(args, num_cus, mfma_gemm::Model::kInt8) != mfma_gemm::Tile::k64x64 ||
      (flip && args.k_bytes % 128 != 0))
    return hipErrorInvalidValue;
  if (args.ep.lhs_sums || args.ep.rhs_sums || (!args.fuse_sums && (args.ep.lhs_zero_point || args.ep.rhs_zero_point)))
    return hipErrorInvalidValue;  // sums arrays are per product: only the fused form is batched
  if (flip) {
    return args.fuse_sums ? mfma_gemm::LaunchSmallestTileBatch<Int8Traits, true, true>(stream, args, batch, count)
                          : mfma_gemm::LaunchSmallestTileBatch<Int8Traits, false, true>(stream, args, batch, count);
  }
  return args.fuse_sums ? mfma_gemm::LaunchSmallestTileBatch<Int8Traits, true>(stream, args, batch, count)
                        : mfma_gemm::LaunchSmallestTileBatch<Int8Traits>(stream, args, batch, count);
}

}  // namespace ruyamd
