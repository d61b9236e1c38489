// The GEMM on 32x32 tiles (small_gemm.h) for 8-bit operands.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "int8_traits.h"
#include "small_gemm.h"

namespace ruyamd {
namespace {

struct Int8Small {
  using Acc = mfma_gemm::v16i;
  using Value = int;
  static constexpr int kElementA = 1, kElementB = 1;
  static __device__ __forceinline__ void Mma(const v4i& a, const v4i& b, Acc (&acc)[1], int) {
    Mma(a, b, acc[0]);
  }
  static __device__ __forceinline__ void Mma(const v4i& a, const v4i& b, Acc& acc) {
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, acc, 0, 0, 0);
  }
  static __device__ __forceinline__ int Bits(int x) { return x; }
  static __device__ __forceinline__ int FromBits(int x) { return x; }

  // Of one row or column: bias, the other side's zero point's share if its sums
  // are at hand, multiplier and exponent if the channels run that way.
  struct Params {
    int32_t bias, sum, m, e;
  };
  static __device__ __forceinline__ void LoadParams(const Epilogue& ep, bool is_row, int index, Params& p) {
    const bool channel = is_row != (ep.channel_is_col != 0);
    const int32_t* sums = is_row ? ep.lhs_sums : ep.rhs_sums;
    p.bias = channel && ep.bias ? static_cast<const int32_t*>(ep.bias)[index] : 0;
    p.sum = (is_row ? ep.rhs_zero_point : ep.lhs_zero_point) && sums ? sums[index] : 0;
    p.m = channel && ep.mult_fixedpoint ? ep.mult_fixedpoint[index] : ep.mult_fixedpoint_scalar;
    p.e = channel && ep.mult_fixedpoint ? ep.mult_exponent[index] : ep.mult_exponent_scalar;
  }
  static __device__ __forceinline__ void StageParams(const Epilogue& ep, bool is_row, const Params& p, int* at, int stride) {
    const uint32_t zero_point = static_cast<uint32_t>(is_row ? ep.rhs_zero_point : ep.lhs_zero_point);
    at[0] = static_cast<int32_t>(static_cast<uint32_t>(p.bias) - zero_point * static_cast<uint32_t>(p.sum) +
                                 (is_row ? static_cast<uint32_t>(ep.zp_product_depth) : 0u));
    at[stride] = p.m;
    at[2 * stride] = p.e;
  }
  static __device__ __forceinline__ void Finish(const int (&total)[4], const int* area, int stride, int row, int col,
                                                const Epilogue& ep, int (&vals)[4]) {
    const int column_add = area[col];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      vals[e] = static_cast<int>(static_cast<uint32_t>(total[e]) + static_cast<uint32_t>(area[row + e]) +
                                 static_cast<uint32_t>(column_add));
    if (ep.requantize && !ep.mult_fixedpoint && ep.mult_exponent_scalar <= -2) {
      const int high_shift = -1 - ep.mult_exponent_scalar;  // (31 - e) - 32
#pragma unroll
      for (int e = 0; e < 4; ++e) vals[e] = RequantHigh(vals[e], ep.mult_fixedpoint_scalar, high_shift);
    } else if (ep.requantize) {
      if (ep.channel_is_col) {
        const int m = area[stride + col], exponent = area[2 * stride + col];
#pragma unroll
        for (int e = 0; e < 4; ++e) vals[e] = MultiplyByQuantizedMultiplier(vals[e], m, exponent);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          vals[e] = MultiplyByQuantizedMultiplier(vals[e], area[stride + row + e], area[2 * stride + row + e]);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      vals[e] = Median3(static_cast<int32_t>(static_cast<uint32_t>(vals[e]) + static_cast<uint32_t>(ep.dst_zero_point)),
                        ep.clamp_min_i, ep.clamp_max_i);
  }
};

// int8 x int16, the int16 operand's planes formed on the way to LDS: neither a
// pack launch nor, whichever side it is, a destination to be reordered. What the
// low plane lacks is 128 times the sum of the int8 vector (a zero point of -128,
// which the dispatcher hands over as the fused factor).
struct Int8Int16Small : Int8Small {
  static constexpr int kElementA = 1, kElementB = 2;
};
struct Int16Int8Small : Int8Small {
  static constexpr int kElementA = 2, kElementB = 1;
};

// Whether an operand's runs do not all start at multiples of 16 bytes. Across the
// vectors, 16-byte loads of such runs cost what those at odd addresses do (1000^3,
// int8 transposed, int16 along the rows: 12.7 us expected, 21.2 measured).
bool Straddling(const GemmArgs& args) {
  return ((reinterpret_cast<uintptr_t>(args.a) | reinterpret_cast<uintptr_t>(args.b) | static_cast<uint32_t>(args.lda) |
           static_cast<uint32_t>(args.ldb)) & 15) != 0;
}

}  // namespace

// What the tiles of 32x32 win on is the time that does not depend on the work:
// no pack launch (2.5 us and more), a quarter of the loads, of the adding up and
// of the write-back of a 64x64 tile to a workgroup. What they lose is reuse: they
// read an operand byte twice as often; the form with 64x64 tiles and the depth
// dealt to eight waves lies in between where operands would have to be packed. So
// the lines run along tiles to a CU (a_cu: of 32x32), with limits on the depth from
// where the sides met on a grid of 64 to 2048 tiles and depths of 64 to 8192, three
// sets of buffers in turn (us, other route -> this):
//   used in place: 256 tiles x 512 5.3 -> 4.5, x 1024 6.9 -> 4.8, x 4096 10.8 -> 8.2;
//     512 x 288 4.8 -> 5.0, x 1024 6.9 -> 5.7, x 2048 8.1 -> 7.8, x 4096 11.1 -> 11.3; 768 x
//     1024 6.9 -> 6.8, x 1504 7.7 -> 9.2; 1024 x 512 5.5 -> 6.5.
//   packed by rows otherwise: 256 x 289 6.2 -> 4.9, x 2049 13.6 -> 7.6, x 5697 17.2 ->
//     12.3; 512 x 1025 11.4 -> 7.9, x 2049 13.9 -> 10.6, x 4097 15.8 -> 16.7; 768 x 1025
//     11.6 -> 9.4, x 1505 12.5 -> 10.9, on 64x64 x 2049 13.3 -> 13.0; 1024 x 289 6.3 -> 6.6, x
//     1025 11.7 -> 10.8, on 64x64 x 1505 12.5 -> 11.8, x 2049 13.1 -> 14.1.
//   one side transposed, at whole dwords: 256 x 512 8.3 -> 4.6, x 5696 16.7 -> 14.1; 512 x
//     1024 10.1 -> 7.8, x 2048 11.7 -> 10.6, x 4096 15.3 -> 17.7; 768 x 288 7.5 -> 6.4, on
//     64x64 x 1024 10.2 -> 9.0, x 1504 11.8 -> 10.7, x 2048 11.5 -> 11.7; 1024 x 288 7.5 -> 6.8,
//     x 1024 10.3 -> 9.4, x 1504 11.6 -> 11.4; with four waves 2048 x 256 9.0 -> 7.9.
//   ... and at odd bytes: 256 x 1025 11.0 -> 8.5, x 4097 16.3 -> 16.1, x 5697 18.9 -> 19.0;
//     512 x 513 9.0 -> 8.5, on 64x64 x 1025 11.9 -> 10.6, x 1505 12.7 -> 12.0, x 2049 14.0 ->
//     14.9; 768 x 289 8.0 -> 7.2, x 1025 12.5 -> 10.9, x 1505 13.1 -> 13.1; 1024 x 1025 12.7 ->
//     11.2, x 1505 13.0 -> 14.3; with four waves 2048 x 256 9.4 -> 8.8.
// The lines lie at whole numbers of tiles to a CU: a few tiles above one cost what
// the next one costs (in place x 1024, where the others take 6.8 to 6.9: 768 tiles
// 6.5, 784 7.2, 832 7.5, 1024 7.6). From 769 tiles to 1024, the others -> these:
//   packed by rows: x 129 to 177 5.5 -> 5.0 to 5.1 (whole dwords 5.1 -> 4.7 to 4.8), where
//     some of the four waves have no step; x 193 to 241 5.5 -> 5.4 to 5.6 (5.1 -> 5.0 to
//     5.2); x 257 6.1 -> 6.2 to 6.3, x 513 7.4 -> 7.6, x 769 8.6 -> 8.6 to 8.8, x 961 9.2
//     -> 9.1 to 9.4, x 1025 10.8 -> 9.9 to 10.7, x 1301 11.2 -> 12.5, on 64x64 10.9 to 11.3.
//   one side transposed, whole dwords: x 200 7.3 -> 5.6 on either, x 288 7.5 -> 6.6, on 64x64
//     6.3, x 1408 11.0 -> 10.4, x 1600 12.1 -> 10.8, x 1792 11.9 -> 11.1.
// Operands that come from HBM (weights in turn, more than the caches hold) are slower
// here at the largest depths unless most CUs have a tile: 2048 x 8192 x 32 (64 tiles) 11.5
// -> 13.2, with one side transposed 14.3 -> 15.9, x 96 (192) 11.9 -> 12.9, 4096 x 8192 x 32
// (128) 13.3 -> 14.0, x 48 (256) 13.7 -> 13.1, 8192 x 8192 x 32 (256) 18.6 -> 16.8.
// More waves to a workgroup, or longer steps, where the grid leaves CUs room for
// them: 256 tiles in place x 4096 8.8 with four waves, 8.2 with eight; packed x 4097
// 12.9 and 10.4; transposed x 4096 11.3 with eight, 10.6 with sixteen.
SmallGemmPlan PlanSmallGemmI8(const GemmArgs& args, int num_cus, SmallGemmPlan plan, uint64_t packed_bytes) {
  const int64_t tiles = int64_t((args.M + 31) / 32) * ((args.N + 31) / 32);
  const int64_t tiles64 = int64_t((args.M + 63) / 64) * ((args.N + 63) / 64);
  const int K = args.k_valid;
  const bool across = small_gemm::IsAcross(plan.source_a) || small_gemm::IsAcross(plan.source_b);
  const bool bytes = small_gemm::IsAnyByte(plan.source_a) || small_gemm::IsAnyByte(plan.source_b) ||
                     (across && Straddling(args));
  const int a_cu = tiles <= num_cus ? 1 : tiles <= 2 * num_cus ? 2 : tiles <= 3 * num_cus ? 3 : tiles <= 4 * num_cus ? 4 : 8;
  plan.waves = 0;
  if (tiles > 8 * num_cus || K < 16) return plan;
  // Depths in [from32, to32] are for the 32x32 tiles, above that to to64 for the
  // 64x64 ones.
  int from32 = 16, to32 = 0, to64 = 0;
  const int deepest = 4 * tiles <= 3 * num_cus ? 7680 : 8192;
  if (across) {
    to32 = a_cu == 1 ? (bytes ? 4352 : deepest) : a_cu == 2 ? (bytes ? 700 : 2560) : a_cu == 3 ? (bytes ? 200 : 400) : a_cu == 4 ? 200 : 0;
    to64 = a_cu == 1 ? 0 : a_cu == 2 ? (bytes ? 1600 : 0) : a_cu <= 4 ? (bytes ? 1250 : 1800) : 300;
  } else if (packed_bytes) {
    from32 = a_cu == 4 && K > 192 ? 960 : 16;
    to32 = a_cu == 1 ? 8192 : a_cu == 2 ? 2560 : a_cu == 3 ? 1536 : a_cu == 4 ? 1300 : 0;
    to64 = a_cu == 4 ? 1700 : 0;
  } else {
    from32 = a_cu == 1 ? 16 : a_cu == 2 ? 448 : 700;
    to32 = a_cu == 1 ? deepest : a_cu == 2 ? 3072 : a_cu == 3 ? 1088 : 0;
  }
  if (K < from32) return plan;
  if (K > to32) {
    if (K > to64 || tiles64 > 2 * num_cus) return plan;
    plan.tile = 64;
    plan.waves = tiles64 <= num_cus ? 8 : 4;
    plan.step = 64;
    return plan;
  }
  plan.waves = 4;
  plan.step = 64;
  if (across) {
    if (a_cu == 1) {
      plan.waves = K >= 4096 ? (bytes ? 4 : 16) : K > 256 ? 8 : 4;
      if (K > 256) plan.step = 128;
    } else if (a_cu == 2) {
      plan.step = 128;
    }
  } else if (a_cu == 1) {
    // (In place, 256 tiles: x 512 4.64 with four waves, 4.54 with eight; x 1024 4.83
    // and 5.17; x 1504 5.89 and 6.18; x 2048 6.21 and 5.97; x 4096 8.77 and 8.18. Deep rows that
    // come from beyond L2 want more bytes in flight: eight waves, then sixteen on
    // longer steps, 99 tiles x 4992 7.8 and 8.3, x 7312 12.9 and 11.6 (12.6 with the
    // depth split on the larger tiles); 64 x 6144 10.4 and 9.5; 128 x 6016 9.6 and 9.4.)
    if (K > 256 && (packed_bytes || K <= 768 || K > 1792)) plan.waves = 8;
    if (!packed_bytes && K > 5760) {
      plan.waves = 16;
      plan.step = 128;
    }
  } else if (bytes && a_cu == 2 && K > 128 && K < 1024) {
    plan.waves = 8;
  }
  return plan;
}

hipError_t LaunchSmallGemmI8(hipStream_t stream, const GemmArgs& args, const SmallGemmPlan& plan) {
  return small_gemm::LaunchPlan<Int8Small>(stream, args, plan);
}

// Held against the other tiles' timing model as in fp32; what has to be packed,
// split into planes or reordered for those costs them two to four launches.
// This side is a fit to 16 to 4096 tiles and depths of 32 to 4096, where it takes
// 3.9 us, 0.7 us (1.2) for every tile a CU has beyond the first, and to a KiB of
// depth and tile 1.4 us on aligned rows, more where operands are transposed
// or lie at odd addresses. us per call, other route -> this: in place, 256 tiles x 512 6.5 -> 4.2,
// x 4096 13.3 -> 8.9, 1024 (one round of 64x64) x 512 7.0 -> 8.3, 1152 x 512 11.7 -> 8.7, 2440 x
// 1024 21.6 -> 18.9, 4096 x 1024 23.3 -> 31.2; rows of odd length, 256 x 1025 15.3 -> 7.2, 2440
// x 1025 32.7 -> 29.9; int8 transposed 256 x 1024 10.6 -> 6.2; int16 transposed, its side
// along the rows, 256 x 1024 14.4 -> 5.9, 2440 x 1024 33.4 -> 23.0; both transposed 256 x
// 1024 16.9 -> 6.7. Of 700 products around the line 24 of 585 on these tiles were slower
// there, by up to a third (448 x 3764 x 2816, rows of odd length, 38 -> 53; 1112 x 1888 x
// 1536 with the int16 side transposed 24.6 -> 31.0), with 1.7 and 1.45 us for aligned
// transposed operands and no margin against the 128x128 tile. Set as they are, 11 of
// 558 are, by a fifth at most. A side of up to three tiles has the other operand read
// once, and one of 16 MB and more from HBM where weights take turns: 1.95 us to a KiB of
// depth then (4096 x 8192 x 32 17.4 -> 20.3, 8192 x 4096 x 64 17.4 -> 19.2, 4096 x 4096 x 96
// 15.2 -> 16.6, but 8192 x 4096 x 32 16.1 -> 13.9, 4096 x 4096 x 64 14.5 -> 12.2).
SmallGemmPlan PlanSmallGemmI8I16(const GemmArgs& args, int num_cus, SmallGemmPlan plan, int packs, uint64_t packed_bytes,
                                 bool int16_is_a) {
  const int64_t tiles = int64_t((args.M + 31) / 32) * ((args.N + 31) / 32);
  const int K = args.k_valid;
  plan.waves = 0;
  if (K < 16 || tiles > 10 * num_cus) return plan;
  const bool across8 = small_gemm::IsAcross(int16_is_a ? plan.source_b : plan.source_a);
  const bool across16 = small_gemm::IsAcross(int16_is_a ? plan.source_a : plan.source_b);
  const bool straddling = Straddling(args);
  const bool bytes = small_gemm::IsAnyByte(plan.source_a) || small_gemm::IsAnyByte(plan.source_b) ||
                     (straddling && (across8 || across16));
  const int a_cu = static_cast<int>((tiles + num_cus - 1) / num_cus);
  const bool streamed = std::min(args.M, args.N) <= 96 && int64_t(std::max(args.M, args.N)) * K >= 16000000;
  const double to_a_kib = bytes      ? (across8 || across16 ? 3.4 : 2.4)
                          : across8  ? (across16 ? 2.3 : 1.9)
                          : across16 ? 1.6
                          : streamed ? 1.95
                                     : straddling ? 1.8 : 1.4;
  const double here = 3.9 + (bytes && (across8 || across16) ? 1.2 : 0.7) * (a_cu - 1) + to_a_kib * a_cu * K / 1024.0;
  // (The model counts plane vectors, 64 to 32 columns, with the int8 side along the rows.)
  GemmArgs planes = args;
  planes.M = int16_is_a ? args.N : args.M;
  planes.N = ((int16_is_a ? args.M : args.N) + 31) / 32 * 64;
  const mfma_gemm::TimingModel model = mfma_gemm::TimingModelOf(mfma_gemm::Model::kInt8PlaneSplit);
  const double pack = packs ? 0.5 + 2.0 * packs + 0.7e-6 * static_cast<double>(packed_bytes) : 0;
  for (int i = 0; i < model.count; ++i) {
    // (Deep products on the 128x128 tile with packs in front are over- and these tiles
    // underestimated a little, other than those that transpose at odd addresses.)
    const bool large = model.tiles[i].bm == 128 && model.tiles[i].bn == 128 && !(bytes && (across8 || across16));
    const double other = mfma_gemm::ModelledMicroseconds(planes, num_cus, model, model.tiles[i]) + pack;
    if (here >= (large ? 0.92 : 1.0) * other) return plan;
  }
  plan.waves = a_cu == 1 && K >= 256 ? 8 : 4;
  plan.step = 64;
  return plan;
}

hipError_t LaunchSmallGemmI8I16(hipStream_t stream, const GemmArgs& args, const SmallGemmPlan& plan, bool int16_is_a) {
  return int16_is_a ? small_gemm::LaunchPlan<Int16Int8Small>(stream, args, plan)
                    : small_gemm::LaunchPlan<Int8Int16Small>(stream, args, plan);
}

}  // namespace ruyamd
