// Pack and sums kernels: the device counterpart of the reference's packing
// stage (generic ruy/pack.h:105-132; AVX-512 ruy/pack_avx512.cc:840-1098).
// Packing re-lays an operand out as depth-contiguous int8 vectors (the operand
// order of the int8 matrix instructions), converts uint8 to int8 by flipping
// the top bit (ruy/pack_common.h:36-58), zero-fills the depth padding, and
// produces the per-vector int32 sums that the zero-point correction needs.
// Operands that already have that layout are used in place and only summed.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../internal.h"
#include "gemm_i8.h"
#include "granule.h"
#include "pack.h"

namespace ruyamd {
namespace {

using granule::LoadGranule;
using granule::LowBytes;
using granule::PlaceGranule;
using granule::v4i;
typedef uint32_t UnalignedU32 __attribute__((aligned(1)));

constexpr int kThreads = 256;
constexpr int kTileC = 64;  // transposed 8-bit source: vectors per block
constexpr int kTileK = 64;  // ... and depth bytes per step
constexpr int kPitch = kTileK + 4;  // LDS row pitch in bytes (breaks bank alignment)
constexpr int kTile32 = 32;  // transposed fp32 source: vectors per block and depth positions per step

__device__ __forceinline__ int WaveSum(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// How a launch packs one operand: depth-contiguous rows with 16 or 64 lanes to
// a row, or a transposed source. Compile-time, so that a kernel holds nothing
// but what it needs (these kernels run for a microsecond or two: fetching the
// instructions of the other kinds, a division by a lane count and a shuffle
// loop of unknown length cost them a third of that).
enum PackKind { kNone, kRows16, kRows64, kTranspose8, kTranspose32, kPackKinds };
struct PackPlan {
  PackKind kind = kNone;
  int32_t blocks_c = 0;        // workgroups along the vectors ...
  int32_t parts = 1;           // ... and along the depth
  int32_t depth = 0;           // bytes of a packed vector, to the end of its last granule
  int32_t k_span = 0;          // depth bytes (fp32: positions) of a part
};

// Depth-contiguous source of any alignment and depth (8-bit or fp32: bytes are
// moved): kLanes lanes to a vector, four granules of a lane in flight. (Rows of
// less than a granule are a case of their own, kShort: a fork in front of each
// load made the compiler await the first before it issued the next, and the
// packing of 294 rows of 864 bytes took 4.1 us instead of 3.3.)
template <int kLanes, bool kShort>
__device__ __forceinline__ void PackRowsOf(const PackJob& job, int depth, int k_span, int bx, int by) {
  constexpr int kStep = kLanes * 16;
  const int lane = threadIdx.x % kLanes;
  const int c = bx * (kThreads / kLanes) + static_cast<int>(threadIdx.x / kLanes);
  const bool exists = c < job.src.count;
  const int element = job.src.dtype == RUYAMD_DTYPE_F32 ? 4 : 1;
  const int bytes = job.src.K * element;
  const uint8_t* row =
      static_cast<const uint8_t*>(job.src.data) + int64_t(min(c, job.src.count - 1)) * job.src.stride_c * element;
  const uint32_t flip = job.src.dtype == RUYAMD_DTYPE_U8 ? 0x80808080u : 0u;
  const int k_end = min(depth, (by + 1) * k_span);
  const int end = min(k_end, bytes);
  char* out = static_cast<char*>(job.dst) + int64_t(c) * job.ld;
  constexpr int kInFlight = kShort ? 1 : 4;
  int sum = 0;
  for (int base = by * k_span; base < k_end; base += kInFlight * kStep) {
    v4i x[kInFlight];
#pragma unroll
    for (int i = 0; i < kInFlight; ++i)
      if (i == 0 || base + i * kStep < end) x[i] = LoadGranule<kShort>(row, base + i * kStep + lane * 16, bytes);  // (uniform)
#pragma unroll
    for (int i = 0; i < kInFlight; ++i) {
      if (i > 0 && base + i * kStep >= end) break;
      const int k = base + i * kStep + lane * 16;
      x[i] = PlaceGranule<kShort>(x[i], k, bytes);
      if (flip) {  // (the padding stays zero)
#pragma unroll
        for (int d = 0; d < 4; ++d) x[i][d] ^= static_cast<int>(flip & LowBytes(bytes - k - 4 * d));
      }
      if (exists && k < k_end) *reinterpret_cast<v4i*>(out + k) = x[i];
      // (Granules at k_end and beyond: zero, or of a depth in parts, which has no sums.)
#pragma unroll
      for (int d = 0; d < 4; ++d) sum = __builtin_amdgcn_sdot4(x[i][d], 0x01010101, sum, false);
    }
  }
  if (job.sums) {
#pragma unroll
    for (int off = kLanes / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if (exists && lane == 0) job.sums[c] = sum;
  }
}
template <int kLanes>
__device__ __forceinline__ void PackRows(const PackJob& job, int depth, int k_span, int bx, int by) {
  const int bytes = job.src.K * (job.src.dtype == RUYAMD_DTYPE_F32 ? 4 : 1);
  if (kLanes == 64 || bytes >= 16)  // (64 lanes only take rows beyond 1 KiB: PlanOf)
    PackRowsOf<kLanes, false>(job, depth, k_span, bx, by);
  else
    PackRowsOf<kLanes, true>(job, depth, k_span, bx, by);
}

// 8-bit source contiguous along the vectors (the transposed case), base and
// pitch of any alignment (global loads take any byte address on this target;
// with an odd pitch the dword loads are merely slower than aligned ones): a
// block moves a 64-vector x 64-depth tile per step.
// Each thread loads four dwords (4 vectors x 4 consecutive depth positions),
// transposes the 4x4 bytes in registers with v_perm_b32 and writes four
// dwords to the LDS tile, from which the block writes depth-contiguous
// 16-byte pieces.
__device__ __forceinline__ void PackTranspose8(const PackJob& job, int depth, int k_span, int bx, int by, uint8_t* tile) {
  const PackSource& src = job.src;
  const int tid = threadIdx.x;
  const int c0 = bx * kTileC;
  const int ld = job.ld;
  const int k_begin = by * k_span;
  const int k_end = min(k_begin + k_span, depth);
  const uint8_t* s = static_cast<const uint8_t*>(src.data);
  int8_t* dst = static_cast<int8_t*>(job.dst);
  const uint32_t flip = src.dtype == RUYAMD_DTYPE_U8 ? 0x80808080u : 0u;
  const int cq = tid & 15;   // quad of vectors
  const int kq = tid >> 4;   // quad of depth positions
  const int wc = tid >> 2;   // writer role: vector wc, 16-byte granule wg
  const int wg = tid & 3;
  int32_t sum = 0;
  for (int k0 = k_begin; k0 < k_end; k0 += kTileK) {
    uint32_t r[4];
    const int cfirst = c0 + cq * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + kq * 4 + i;
      r[i] = 0u;
      if (k < src.K) {
        const uint8_t* at = s + int64_t(k) * src.stride_k + cfirst;
        if (cfirst + 4 <= src.count) {
          r[i] = *reinterpret_cast<const UnalignedU32*>(at);
        } else {
          // The last vectors of a count that is not a multiple of four: nothing is read past the row's end.
          for (int j = 0; cfirst + j < src.count; ++j) r[i] |= uint32_t(at[j]) << (8 * j);
        }
      }
    }
    // 4x4 byte transpose: t[j] = depth bytes k..k+3 of vector cfirst + j.
    const uint32_t x0 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);
    const uint32_t x1 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
    const uint32_t y0 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
    const uint32_t y1 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
    uint32_t t[4];
    t[0] = __builtin_amdgcn_perm(y0, x0, 0x05040100u);
    t[1] = __builtin_amdgcn_perm(y0, x0, 0x07060302u);
    t[2] = __builtin_amdgcn_perm(y1, x1, 0x05040100u);
    t[3] = __builtin_amdgcn_perm(y1, x1, 0x07060302u);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<uint32_t*>(tile + (cq * 4 + j) * kPitch + kq * 4) = t[j];
    __syncthreads();
    const int c = c0 + wc;
    const int k = k0 + wg * 16;
    if (c < src.count && k < depth) {
      const uint32_t* row = reinterpret_cast<const uint32_t*>(tile + wc * kPitch + wg * 16);
      v4i out;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t w = row[d] ^ (flip & LowBytes(src.K - k - 4 * d));
        out[d] = static_cast<int>(w);
        sum = __builtin_amdgcn_sdot4(static_cast<int>(w), 0x01010101, sum, false);
      }
      *reinterpret_cast<v4i*>(dst + int64_t(c) * ld + k) = out;
    }
    __syncthreads();
  }
  if (job.sums) {
    // The four granule writers of a vector are adjacent lanes.
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    const int c = c0 + wc;
    if (wg == 0 && c < src.count) job.sums[c] = sum;
  }
}

// The same for fp32: 32 vectors x 32 depth positions per step through LDS.
// There are no sums and no conversion for floating point
// (ruy/pack_common.h:100-133).
__device__ __forceinline__ void PackTranspose32(const PackJob& job, int depth_bytes, int k_span, int bx, int by,
                                                float (*tile)[kTile32 + 1]) {
  const PackSource& src = job.src;
  const int tx = threadIdx.x & 31;
  const int ty = threadIdx.x >> 5;  // 0..7
  const int c0 = bx * kTile32;
  const int ld = job.ld / 4, depth = depth_bytes / 4;
  const float* s = static_cast<const float*>(src.data);
  float* dst = static_cast<float*>(job.dst);
  const int k_end = min(depth, (by + 1) * k_span);
  for (int k0 = by * k_span; k0 < k_end; k0 += kTile32) {
#pragma unroll
    for (int t = ty; t < kTile32; t += 8) {
      const int c = c0 + tx;
      const int k = k0 + t;
      float v = 0.f;
      if (c < src.count && k < src.K) v = s[c + k * src.stride_k];
      tile[tx][t] = v;
    }
    __syncthreads();
#pragma unroll
    for (int t = ty; t < kTile32; t += 8) {
      const int c = c0 + t;
      const int k = k0 + tx;
      if (c < src.count && k < depth) dst[int64_t(c) * ld + k] = tile[t][tx];
    }
    __syncthreads();
  }
}

// Both operands of a product in one launch: a second one would cost more than
// the packing of all but the largest. Where the depth of a vector is dealt to
// several workgroups nobody forms its sums here (adding the parts up took a
// launch in front that cleared the words): the product does, as for operands
// used in place. Calls with both packed, as up to four launches in front of the
// product -> as one: 1000 x 1500 x 700 int8 with one side transposed 20.4 ->
// 13.0 us, 64 x 147 x 12544 uint8 13.5 -> 9.8 us, 256 x 1968 x 645 uint8 20.9 ->
// 13.8 us. The first `first` workgroups take the first operand.
struct PackLaunch {
  PackJob job[2];
  int32_t blocks_c[2];
  int32_t depth[2];
  int32_t k_span[2];
  int32_t first;  // workgroups of the first operand
};
template <int kKind>
__device__ __forceinline__ void PackOperand(const PackJob& job, int depth, int k_span, int blocks_c, int block, void* tile) {
  const int by = block < blocks_c ? 0 : block / blocks_c;
  const int bx = block - by * blocks_c;
  if constexpr (kKind == kRows16) PackRows<16>(job, depth, k_span, bx, by);
  if constexpr (kKind == kRows64) PackRows<64>(job, depth, k_span, bx, by);
  if constexpr (kKind == kTranspose8) PackTranspose8(job, depth, k_span, bx, by, static_cast<uint8_t*>(tile));
  if constexpr (kKind == kTranspose32)
    PackTranspose32(job, depth, k_span, bx, by, static_cast<float(*)[kTile32 + 1]>(tile));
}
constexpr int TileBytes(int kind) {
  return kind == kTranspose8 ? kTileC * kPitch : kind == kTranspose32 ? kTile32 * (kTile32 + 1) * 4 : 16;
}
template <int kFirst, int kSecond>
__global__ __launch_bounds__(kThreads) void PackKernel(PackLaunch launch) {
  constexpr int kBytes = TileBytes(kFirst) > TileBytes(kSecond) ? TileBytes(kFirst) : TileBytes(kSecond);
  __shared__ __attribute__((aligned(16))) char tile[kBytes];
  const int block = blockIdx.x;
  if (kSecond == kNone || block < launch.first)
    PackOperand<kFirst>(launch.job[0], launch.depth[0], launch.k_span[0], launch.blocks_c[0], block, tile);
  else
    PackOperand<kSecond>(launch.job[1], launch.depth[1], launch.k_span[1], launch.blocks_c[1], block - launch.first, tile);
}

// The kernel for two kinds (operands of one product have one element size).
using PackFunction = void (*)(PackLaunch);
template <int kFirst>
PackFunction KernelFor(PackKind second) {
  constexpr int kTransposed = kFirst == kTranspose32 ? kTranspose32 : kTranspose8;
  switch (second) {
    case kNone:
      return PackKernel<kFirst, kNone>;
    case kRows16:
      return PackKernel<kFirst, kRows16>;
    case kRows64:
      return PackKernel<kFirst, kRows64>;
    case kTranspose32:
      if constexpr (kFirst == kRows16 || kFirst == kRows64) return PackKernel<kFirst, kTranspose32>;
      [[fallthrough]];
    default:
      return second == kTransposed ? PackKernel<kFirst, kTransposed> : nullptr;
  }
}
PackFunction KernelFor(PackKind first, PackKind second) {
  switch (first) {
    case kRows16:
      return KernelFor<kRows16>(second);
    case kRows64:
      return KernelFor<kRows64>(second);
    case kTranspose8:
      return KernelFor<kTranspose8>(second);
    case kTranspose32:
      return KernelFor<kTranspose32>(second);
    default:
      return nullptr;
  }
}

// Parts of a depth of `steps` steps so that some `blocks_wanted` workgroups
// are in flight, each with at least one step; returns the steps of a part.
int StepsPerPart(int steps, int blocks_c, int blocks_wanted, int* parts) {
  int wanted = std::min(steps, std::max(1, (blocks_wanted + blocks_c - 1) / blocks_c));
  const int per_part = (steps + wanted - 1) / wanted;
  *parts = (steps + per_part - 1) / per_part;
  return per_part;
}

PackPlan PlanOf(const PackSource& src) {
  PackPlan plan;
  const int32_t bytes = src.K * (src.dtype == RUYAMD_DTYPE_F32 ? 4 : 1);
  const int32_t depth = plan.depth = bytes > 16 ? (bytes + 15) / 16 * 16 : 16;
  if (src.stride_k == 1) {
    // 16 lanes to a row of up to 1 KiB (what they have in flight at a time).
    plan.kind = depth <= 1024 ? kRows16 : kRows64;
    const int lanes = plan.kind == kRows16 ? 16 : 64;
    const int rows_per_block = kThreads / lanes;
    plan.blocks_c = (src.count + rows_per_block - 1) / rows_per_block;
    // A vector of up to twice what its lanes have in flight is walked in one
    // place (the sums come with it), and so is any when there are a thousand
    // waves; otherwise the depth is dealt out, a granule a lane (1 KiB) at
    // least. So it is for a handful of vectors (the narrow side of a skinny
    // product: 10 x 7805 int8 4.3 us in 3 workgroups, 1.8 in 24).
    const int step = lanes * 16;
    const int steps = (depth + step - 1) / step;
    int per_part = steps;
    if ((steps > 8 && plan.blocks_c < 256) || plan.blocks_c < 16)
      per_part = StepsPerPart(steps, plan.blocks_c, 512, &plan.parts);
    plan.k_span = per_part * step;
  } else if (src.dtype == RUYAMD_DTYPE_F32) {
    plan.kind = kTranspose32;
    plan.blocks_c = (src.count + kTile32 - 1) / kTile32;
    plan.k_span = kTile32 * StepsPerPart((depth / 4 + kTile32 - 1) / kTile32, plan.blocks_c, 4096, &plan.parts);
  } else {
    plan.kind = kTranspose8;
    plan.blocks_c = (src.count + kTileC - 1) / kTileC;
    // A block's steps are a chain of load, transposition through LDS and store
    // (about a microsecond each), so a block gets as few of them as some two
    // thousand blocks allow (a 2048 x 2048 operand: 7.2 -> 3.6 us); one or two
    // stay together, and the sums come with them.
    const int steps = (depth + kTileK - 1) / kTileK;
    int per_part = steps;
    if (steps > 2) per_part = StepsPerPart(steps, plan.blocks_c, 2048, &plan.parts);
    plan.k_span = per_part * kTileK;
  }
  return plan;
}

// One wave per vector, 16 bytes per lane per step.
// `flip` = 0x80808080 for uint8 data used in place (value - 128 is the byte
// with its top bit flipped, read as int8), 0 for int8 data.
__global__ __launch_bounds__(256) void SumsI8Kernel(const int8_t* data, int32_t ld, int32_t count,
                                                   int32_t K, int32_t* sums, int32_t flip) {
  const int lane = threadIdx.x & 63;
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= count) return;
  const int8_t* row = data + int64_t(c) * ld;
  int32_t s0 = 0, s1 = 0;
  int k = lane * 16;
  for (; k + 1024 < K; k += 2048) {
    const v4i x = *reinterpret_cast<const v4i*>(row + k);
    const v4i y = *reinterpret_cast<const v4i*>(row + k + 1024);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      s0 = __builtin_amdgcn_sdot4(x[d] ^ flip, 0x01010101, s0, false);
      s1 = __builtin_amdgcn_sdot4(y[d] ^ flip, 0x01010101, s1, false);
    }
  }
  for (; k < K; k += 1024) {
    const v4i x = *reinterpret_cast<const v4i*>(row + k);
#pragma unroll
    for (int d = 0; d < 4; ++d) s0 = __builtin_amdgcn_sdot4(x[d] ^ flip, 0x01010101, s0, false);
  }
  const int32_t total = WaveSum(s0 + s1);
  if (lane == 0) sums[c] = total;
}

// int16 -> two int8 planes. Block = 32 vectors (one group) x a depth span; the
// 32x32 int16 tile goes through LDS so reads follow the source's contiguous
// dimension; each thread then emits 4 consecutive depth bytes of one plane.
__global__ __launch_bounds__(256) void PackI16SplitKernel(PackSource src, int8_t* dst, int32_t ld) {
  __shared__ int16_t tile[32][33];
  const int tx = threadIdx.x & 31;
  const int ty = threadIdx.x >> 5;  // 0..7
  const int group = blockIdx.x;
  const int c0 = group * 32;
  const int16_t* s = static_cast<const int16_t*>(src.data);
  const bool depth_contiguous = src.stride_k == 1;
  for (int k0 = blockIdx.y * 32; k0 < ld; k0 += gridDim.y * 32) {
#pragma unroll
    for (int t = ty; t < 32; t += 8) {
      const int c = c0 + (depth_contiguous ? t : tx);
      const int k = k0 + (depth_contiguous ? tx : t);
      int16_t v = 0;
      bool real = c < src.count && k < src.K;
      if (real) v = s[c * src.stride_c + k * src.stride_k];
      if (depth_contiguous)
        tile[t][tx] = v;
      else
        tile[tx][t] = v;
    }
    __syncthreads();
    // thread -> (vector cc = tid / 8, depth quad kq = tid % 8), both planes
    const int cc = threadIdx.x >> 3;
    const int kq = (threadIdx.x & 7) * 4;
    if (k0 + kq < ld) {
      uint32_t hi = 0, lo = 0;
      const bool real_c = c0 + cc < src.count;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const int k = k0 + kq + d;
        if (real_c && k < src.K) {
          const int v = tile[cc][kq + d];
          hi |= (static_cast<uint32_t>(v >> 8) & 0xffu) << (8 * d);
          lo |= (static_cast<uint32_t>((v & 0xff) - 128) & 0xffu) << (8 * d);
        }
      }
      int8_t* base = dst + (int64_t(group) * 64 + cc) * ld + k0 + kq;
      *reinterpret_cast<uint32_t*>(base) = hi;
      *reinterpret_cast<uint32_t*>(base + int64_t(32) * ld) = lo;
    }
    __syncthreads();
  }
}

// The same split for a depth-contiguous, 16-byte aligned int16 source whose
// depth is a multiple of 16: pure streaming, one wave per vector part, each
// lane turns 16 int16 (two 16-byte loads) into 16 high bytes and 16 low bytes
// with v_perm_b32 (the low plane is the low byte with its top bit flipped).
__global__ __launch_bounds__(256) void PackI16SplitRowsKernel(PackSource src, int8_t* dst, int32_t ld) {
  const int lane = threadIdx.x & 63;
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int count_padded = (src.count + 31) / 32 * 32;  // vectors of the last group that do not exist are zero
  if (c >= count_padded) return;
  int8_t* hi_row = dst + (int64_t(c / 32) * 64 + c % 32) * ld;
  int8_t* lo_row = hi_row + int64_t(32) * ld;
  const int16_t* row = static_cast<const int16_t*>(src.data) + int64_t(c) * src.stride_c;
  for (int k = blockIdx.y * 1024 + lane * 16; k < ld; k += gridDim.y * 1024) {
    v4i hi = {0, 0, 0, 0}, lo = {0, 0, 0, 0};
    if (c < src.count && k < src.K) {
      const v4i x = *reinterpret_cast<const v4i*>(row + k);
      const v4i y = *reinterpret_cast<const v4i*>(row + k + 8);
      hi[0] = __builtin_amdgcn_perm(x[1], x[0], 0x07050301u);
      hi[1] = __builtin_amdgcn_perm(x[3], x[2], 0x07050301u);
      hi[2] = __builtin_amdgcn_perm(y[1], y[0], 0x07050301u);
      hi[3] = __builtin_amdgcn_perm(y[3], y[2], 0x07050301u);
      lo[0] = __builtin_amdgcn_perm(x[1], x[0], 0x06040200u) ^ 0x80808080u;
      lo[1] = __builtin_amdgcn_perm(x[3], x[2], 0x06040200u) ^ 0x80808080u;
      lo[2] = __builtin_amdgcn_perm(y[1], y[0], 0x06040200u) ^ 0x80808080u;
      lo[3] = __builtin_amdgcn_perm(y[3], y[2], 0x06040200u) ^ 0x80808080u;
    }
    *reinterpret_cast<v4i*>(hi_row + k) = hi;
    *reinterpret_cast<v4i*>(lo_row + k) = lo;
  }
}

// dst(i, j) = src(i, j) for two views of the same shape with different storage
// orders, 32x32 elements per block through LDS: reads run along the source's
// contiguous dimension, writes along the destination's.
template <typename T>
__global__ __launch_bounds__(256) void ReorderKernel(const T* src, int64_t src_rs, int64_t src_cs, T* dst,
                                                    int64_t dst_rs, int64_t dst_cs, int rows, int cols) {
  __shared__ T tile[32][33];
  const int tx = threadIdx.x & 31;
  const int ty = threadIdx.x >> 5;  // 0..7
  const int i0 = blockIdx.x * 32;
  const int j0 = blockIdx.y * 32;
  const bool src_rows_contiguous = src_rs == 1;
  const bool dst_rows_contiguous = dst_rs == 1;
#pragma unroll
  for (int t = ty; t < 32; t += 8) {
    const int i = i0 + (src_rows_contiguous ? tx : t);
    const int j = j0 + (src_rows_contiguous ? t : tx);
    if (i < rows && j < cols) tile[i - i0][j - j0] = src[i * src_rs + j * src_cs];
  }
  __syncthreads();
#pragma unroll
  for (int t = ty; t < 32; t += 8) {
    const int i = i0 + (dst_rows_contiguous ? tx : t);
    const int j = j0 + (dst_rows_contiguous ? t : tx);
    if (i < rows && j < cols) dst[i * dst_rs + j * dst_cs] = tile[i - i0][j - j0];
  }
}

}  // namespace

hipError_t LaunchReorder(hipStream_t stream, const DevMat& src, const DevMat& dst) {
  if (dst.rows == 0 || dst.cols == 0) return hipSuccess;
  if ((int64_t(dst.cols) + 31) / 32 > 65535) return hipErrorInvalidValue;  // grid.y
  const dim3 grid((dst.rows + 31) / 32, (dst.cols + 31) / 32);
  switch (DtypeSize(dst.dtype)) {
    case 1:
      hipLaunchKernelGGL(ReorderKernel<uint8_t>, grid, dim3(256), 0, stream, static_cast<const uint8_t*>(src.data),
                         src.rs, src.cs, static_cast<uint8_t*>(dst.data), dst.rs, dst.cs, dst.rows, dst.cols);
      break;
    case 2:
      hipLaunchKernelGGL(ReorderKernel<uint16_t>, grid, dim3(256), 0, stream,
                         static_cast<const uint16_t*>(src.data), src.rs, src.cs, static_cast<uint16_t*>(dst.data),
                         dst.rs, dst.cs, dst.rows, dst.cols);
      break;
    case 4:
      hipLaunchKernelGGL(ReorderKernel<uint32_t>, grid, dim3(256), 0, stream,
                         static_cast<const uint32_t*>(src.data), src.rs, src.cs, static_cast<uint32_t*>(dst.data),
                         dst.rs, dst.cs, dst.rows, dst.cols);
      break;
    case 8:
      hipLaunchKernelGGL(ReorderKernel<uint64_t>, grid, dim3(256), 0, stream,
                         static_cast<const uint64_t*>(src.data), src.rs, src.cs, static_cast<uint64_t*>(dst.data),
                         dst.rs, dst.cs, dst.rows, dst.cols);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t LaunchPackI16Split(hipStream_t stream, const PackSource& src, int8_t* dst, int32_t ld) {
  if (src.count == 0 || ld == 0) return hipSuccess;
  const int groups = (src.count + 31) / 32;
  if (src.stride_k == 1 && src.K % 16 == 0 && (reinterpret_cast<uintptr_t>(src.data) & 15) == 0 &&
      (src.stride_c * 2) % 16 == 0) {
    const int k_blocks = std::min((ld + 1023) / 1024, std::max(1, 2048 / (groups * 32)));
    hipLaunchKernelGGL(PackI16SplitRowsKernel, dim3(groups * 8, k_blocks), dim3(256), 0, stream, src, dst, ld);
    return hipGetLastError();
  }
  int blocks_k = (ld + 31) / 32;
  if (blocks_k > 64) blocks_k = 64;
  hipLaunchKernelGGL(PackI16SplitKernel, dim3(groups, blocks_k), dim3(256), 0, stream, src, dst, ld);
  return hipGetLastError();
}

hipError_t LaunchPack(hipStream_t stream, const PackJob* jobs, int count) {
  PackLaunch launch = {};
  PackKind kinds[2] = {kNone, kNone};
  int used = 0, blocks = 0;
  for (int i = 0; i < count; ++i) {
    const PackJob& job = jobs[i];
    if (job.src.count == 0 || job.ld == 0) continue;
    const PackPlan plan = PlanOf(job.src);
    if (used == 2 || job.ld % 16 != 0 || (job.src.stride_k != 1 && job.src.stride_c != 1) ||
        (job.sums && !PackFormsSums(job.src)))
      return hipErrorInvalidValue;
    launch.job[used] = job;
    launch.blocks_c[used] = plan.blocks_c;
    launch.depth[used] = plan.depth;
    launch.k_span[used] = plan.k_span;
    if (used == 0) launch.first = plan.blocks_c * plan.parts;
    kinds[used] = plan.kind;
    blocks += plan.blocks_c * plan.parts;
    ++used;
  }
  if (used == 0) return hipSuccess;
  const PackFunction kernel = KernelFor(kinds[0], kinds[1]);
  if (!kernel) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), 0, stream, launch);
  return hipGetLastError();
}

bool PackFormsSums(const PackSource& src) {
  return src.dtype != RUYAMD_DTYPE_F32 && (src.count == 0 || PlanOf(src).parts == 1);
}

hipError_t LaunchSumsI8(hipStream_t stream, const int8_t* data, int32_t ld, int32_t count, int32_t K,
                        int32_t* sums, uint32_t flip) {
  if (count == 0) return hipSuccess;
  hipLaunchKernelGGL(SumsI8Kernel, dim3((count + 3) / 4), dim3(256), 0, stream, data, ld, count, K,
                     sums, static_cast<int32_t>(flip));
  return hipGetLastError();
}

}  // namespace ruyamd
