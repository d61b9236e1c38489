// The GEMM on 32x32 tiles (small_gemm.h) for fp32.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mfma_gemm.h"
#include "small_gemm.h"

namespace ruyamd {
namespace {

using granule::v4i;

struct F32Small {
  using Acc = mfma_gemm::v16f;
  using Value = float;
  static constexpr int kElementA = 4, kElementB = 4;
  // A granule holds four consecutive depth values of a vector.
  template <int kChains>
  static __device__ __forceinline__ void Mma(const v4i& a, const v4i& b, Acc (&acc)[kChains], int sub_step) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      Acc& to = acc[kChains == 4 ? sub_step % 2 * 2 + e % 2 : sub_step % kChains];
      to = __builtin_amdgcn_mfma_f32_32x32x2f32(__int_as_float(a[e]), __int_as_float(b[e]), to, 0, 0, 0);
    }
  }
  static __device__ __forceinline__ int Bits(float x) { return __float_as_int(x); }
  static __device__ __forceinline__ float FromBits(int x) { return __int_as_float(x); }

  struct Params {
    float bias;
  };
  static __device__ __forceinline__ void LoadParams(const Epilogue& ep, bool is_row, int index, Params& p) {
    p.bias = is_row != (ep.channel_is_col != 0) && ep.bias ? static_cast<const float*>(ep.bias)[index] : 0.f;
  }
  static __device__ __forceinline__ void StageParams(const Epilogue&, bool, const Params& p, int* at, int) {
    at[0] = __float_as_int(p.bias);
  }
  static __device__ __forceinline__ void Finish(const float (&total)[4], const int* area, int, int row, int col,
                                                const Epilogue& ep, int (&vals)[4]) {
    const float column_bias = __int_as_float(area[col]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = total[e];
      if (ep.bias) v = v + (ep.channel_is_col ? column_bias : __int_as_float(area[row + e]));
      v = ep.clamp_max_f < v ? ep.clamp_max_f : v;
      v = v < ep.clamp_min_f ? ep.clamp_min_f : v;
      vals[e] = __float_as_int(v);
    }
  }
};

}  // namespace

// The time of these tiles by a fit to 16 to 2112 of them and depths of 16 to 2048
// (within 10 % mostly): 3.9 us, 0.33 us for every tile a CU has beyond the first,
// and 1.22 us to a KiB of depth and tile (their matrix instructions alone take 1.03
// at the clock they leave the card), 1.4 where rows do not start at multiples of 16
// bytes or an operand is transposed on the way. Held against the other tiles'
// timing model and a pack in front of them (of transposed operands: rows are read
// in place there, too). us, other route -> this: 512^3 12.8 -> 6.0; 512 tiles in place
// x 512 13.2 -> 8.6, x 2048 23.9 -> 23.5; 1024 x 256 10.6 -> 8.8, x 1024 21.9 -> 23.7; 2112
// (one 64x64 tile too many for two rounds) x 1024 60.5 -> 47.7; 256 tiles with one
// side transposed x 1024 19.7 -> 9.2, both 21.8 -> 9.4; 1536 x 1024 43.4 -> 39.8, both
// 47.6 -> 39.0.
// (Measured against the larger tiles on fp32 instructions. Since two of those run on
// bf16 parts, their model gives them what they are faster at: 860 x 2832 x 1686 80.4 us
// here, 71.1 there; 1024^3 23.7 and 18.3. Held again against every tile for 840 products: by
// these rules 2 % run 5 % or more slower than on the fastest, 4.5 % did by the rules for
// fp32 instructions; 1 %, not 4 %, are over 4 % slower than on those. 205 x 2112 x 352 13.2 us
// here, 15.4 on 64x64 tiles, 1035 x 2288 x 81 14.5 and 16.2, 488 x 1552 x 2336 41.7 and 45.6, 1088 x
// 112 x 2145 with one side transposed 15.4 and 17.4.)
// More than six tiles to a CU: of more than 300 bytes of depth every further one costs
// 0.5 us, with an operand transposed 0.75, and in place the models have to differ by
// more. Of 460 products around the line, 16 to 4096 tiles, these tiles took 392 with
// 0.33 us throughout, of which 31 were slower here (2176 x 288 x 1520 with one side
// transposed 28.0 -> 33.1, 2232 x 1708 x 1352 106 -> 116); they take 354, 10 of them
// slower, by 9 % at most.
// A side of up to three tiles has the other operand read once, and one of 48 MB and
// more comes from beyond the 256 MB of cache that the card has (weights in turn): a
// KiB of depth costs 1.75 us then. 4096 x 4096 x 32 27.4 -> 32.2, 8192 x 2048 x 64 27.7 ->
// 31.0, 8192 x 4096 x 96 69.4 -> 77.1, but 8192 x 2048 x 32 26.7 -> 20.9.
SmallGemmPlan PlanSmallGemmF32(const GemmArgs& args, int num_cus, SmallGemmPlan plan, uint64_t packed_bytes) {
  const int64_t tiles = int64_t((args.M + 31) / 32) * ((args.N + 31) / 32);
  const int K = args.k_valid;
  const bool across = small_gemm::IsAcross(plan.source_a) || small_gemm::IsAcross(plan.source_b);
  plan.waves = 0;
  if (K < 16 || tiles > 16 * num_cus) return plan;
  const int a_cu = static_cast<int>((tiles + num_cus - 1) / num_cus);
  const bool straddling = across || ((reinterpret_cast<uintptr_t>(args.a) | reinterpret_cast<uintptr_t>(args.b) |
                                      static_cast<uint32_t>(args.lda) | static_cast<uint32_t>(args.ldb)) & 15) != 0;
  const bool many = a_cu > 6 && K > 300;
  const bool streamed = !across && std::min(args.M, args.N) <= 96 && int64_t(std::max(args.M, args.N)) * K >= 48000000;
  // (In place in a single round, us to a KiB of depth: 1.13 on few CUs, on all of them 1.33 or, of
  // straddling rows, 1.55.)
  const double filled = static_cast<double>(tiles) / num_cus;
  const double per_kib = streamed               ? 1.75
                         : a_cu == 1 && !across ? 1.13 + (straddling ? 0.42 : 0.2) * filled
                         : straddling           ? 1.4
                                                : 1.22;
  const double here = 3.9 + (!many ? 0.33 : across ? 0.75 : 0.5) * (a_cu - 1) + per_kib * a_cu * K / 1024.0;
  const mfma_gemm::TimingModel model = mfma_gemm::TimingModelOf(mfma_gemm::Model::kF32);
  const double pack = packed_bytes ? 2.3 + 0.5e-6 * static_cast<double>(packed_bytes) : 0;
  // (Many tiles in place on both sides: where the models differ by more than they err. Shallow
  // products of packed operands: the larger tiles err the other way, 1643 x 112 x 1502 16.8 us by
  // their model and 18.8 measured, here 15.4.)
  const double margin = packed_bytes ? (K < 512 ? 1.1 : 1.0) : many ? 0.96 : 1.0;
  for (int i = 0; i < model.count; ++i)
    if (here >= margin * (mfma_gemm::ModelledMicroseconds(args, num_cus, model, model.tiles[i]) + pack)) return plan;
  plan.waves = 4;
  plan.step = 64;
  if (a_cu == 1) {
    plan.waves = K > 256 ? 8 : 4;
    if (across && K >= 1024) plan.step = 128;
    if (across && K >= 4096) plan.waves = 16;
  } else if (across && (K >= 512 || a_cu == 2)) {
    plan.step = 128;
  }
  return plan;
}

hipError_t LaunchSmallGemmF32(hipStream_t stream, const GemmArgs& args, const SmallGemmPlan& plan) {
  return small_gemm::LaunchPlan<F32Small>(stream, args, plan);
}

}  // namespace ruyamd
