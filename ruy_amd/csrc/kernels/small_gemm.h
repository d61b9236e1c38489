// Matrix-core GEMM for products whose run time is that of a launch, a trip to
// memory and a write-back: 32x32 tiles, so that few destination values still
// keep every CU busy, and operands of any layout and alignment read where they
// lie, so that no pack launch stands in front. (8-bit operands also on tiles of
// 64x64, for grids in between that would otherwise need one.)
//
// One workgroup per tile. The depth is dealt to its waves in steps of S bytes:
// wave w takes steps w, w + kWaves, ..., computes the whole tile for them and
// never waits for another wave until the partial tiles are added through LDS.
// The loads of a step go through registers (in flight while the steps before
// are multiplied) into a slot of LDS that is the wave's own, where an operand
// lies depth-contiguous with its 16-byte granules XOR-swizzled by the row
// number, and from there to the matrix instructions. On the way:
//   kSmallRows         rows of depth-contiguous values that start at multiples
//                      of 4 bytes: one 16-byte load a granule;
//   kSmallRowsBytes    ... at any byte: the aligned dwords that hold the
//                      granule, four in one load and the fifth in another,
//                      shifted into place (a 16-byte load at an odd address
//                      takes a CU's address unit four times as long);
//   kSmallAcross       values contiguous along the vectors (the transposed
//                      storage order): a lane loads 16 bytes of vectors at
//                      each of four depth positions and transposes them in its
//                      registers;
//   kSmallAcrossBytes  ... at any byte.
// uint8 data becomes int8 there (the top bit flipped) and what lies past the
// end of the depth zero. Pending depth sums (zero points) come from the
// fragments, a v_dot4 per dword, and are added through LDS like the tiles.
#ifndef RUY_AMD_CSRC_KERNELS_SMALL_GEMM_H_
#define RUY_AMD_CSRC_KERNELS_SMALL_GEMM_H_

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "../epilogue.h"
#include "gemm_i8.h"
#include "granule.h"

namespace ruyamd {
namespace small_gemm {

using granule::LowBytes;
using granule::PlaceGranule;
using granule::v4i;
typedef v4i v4i_dwords __attribute__((aligned(4)));

RUYAMD_HOST_DEVICE constexpr bool IsAcross(int source) {
  return source == kSmallAcross || source == kSmallAcrossBytes;
}
RUYAMD_HOST_DEVICE constexpr bool IsAnyByte(int source) {
  return source == kSmallRowsBytes || source == kSmallAcrossBytes;
}

// Granule g of vector r of a slot whose vectors are S bytes: 16 consecutive
// vectors at one granule index lie in 16 different groups of four banks.
template <int S>
__device__ __forceinline__ int SlotOffset(int r, int g) {
  static_assert(S == 64 || S == 128, "");
  return r * S + ((g ^ (S == 64 ? (r >> 2) & 3 : (r >> 1) & 7)) << 4);
}

// The kTile vectors of one operand that a tile needs, from vector `first` on.
// kElement: bytes of a value. Values of two bytes become two planes of int8, high
// and low byte (minus 128), which lie in the slot one behind the other: v = 256 high
// + low + 128. Across the vectors their bytes are what a piece transposes: byte 2 v
// of a depth position belongs to the low plane of vector v, the next one to the
// high plane.
template <int kTile, int S, int kSource, int kElement>
struct Side {
  static constexpr bool kAcross = IsAcross(kSource);
  static constexpr bool kAnyByte = IsAnyByte(kSource);
  static constexpr bool kPlanes = kElement == 2;
  static constexpr int kSlotVectors = kPlanes ? 2 * kTile : kTile;
  static constexpr int kGranules = S / 16;
  // Bytes of depth that a position takes in a slot, and bytes of source for one
  // of depth along a vector.
  static constexpr int kPosition = kElement == 4 ? 4 : 1;
  static constexpr int kScale = kPlanes ? 2 : 1;
  // Across the vectors: a piece is 16 bytes of them (4 vectors, 16, or the bytes
  // of 8) at four depth positions (4 or 16 bytes of depth).
  static constexpr int kColumnBytes = kElement == 4 ? 4 : 1;  // what is transposed as one
  static constexpr int kColumns = 16 / kColumnBytes;
  static constexpr int kTileColumns = kTile * kScale;
  static constexpr int kPieceDepth = 4 * kPosition;
  static constexpr int kGroups = kTileColumns / kColumns;
  // What a step's work comes to a lane: granules, or pieces.
  static constexpr int kAll = kAcross ? kGroups * (S / kPieceDepth) : kTile * kGranules;
  static constexpr int kUnits = (kAll + 63) / 64;
  static constexpr int kLoads = kAcross ? 4 : kScale;  // of a unit

  const char* data;
  int pitch, count, first, bytes;  // (bytes: of depth in a slot)
  uint32_t flip;
  int lane;
  uint32_t offset[kUnits];  // of the unit's vector (first column)

  struct Held {
    v4i x[kUnits][kLoads];
    int fifth[kUnits][kAnyByte ? kLoads : 1];
  };

  __device__ __forceinline__ bool Exists(int u) const { return kAll % 64 == 0 || u * 64 + lane < kAll; }
  // Vector (first column) of unit u, counted inside the tile, and its first
  // byte of depth, counted inside a step.
  __device__ __forceinline__ int VectorOf(int u) const {
    const int p = u * 64 + lane;
    return kAcross ? p % kGroups * kColumns : p / kGranules;
  }
  __device__ __forceinline__ int DepthOf(int u) const {
    const int p = u * 64 + lane;
    return kAcross ? p / kGroups * kPieceDepth : p % kGranules * 16;
  }
  __device__ __forceinline__ void Start(const void* d, int pitch_, int count_, int first_, int bytes_, uint32_t flip_,
                                        int lane_) {
    data = static_cast<const char*>(d);
    pitch = pitch_;
    count = count_;
    first = first_;
    bytes = bytes_;
    flip = flip_;
    lane = lane_;
    // Vectors past the end read the last one; nothing of them is stored.
    // (Across them: the 16 bytes that end with the last one, moved into place
    // in Store.)
#pragma unroll
    for (int u = 0; u < kUnits; ++u)
      offset[u] = kAcross ? uint32_t(min(first * kScale + VectorOf(u), count * kScale - kColumns) * kColumnBytes)
                          : uint32_t(min(first + VectorOf(u), count - 1)) * uint32_t(pitch);
  }

  // Where load j of unit u of a step reads.
  __device__ __forceinline__ const char* From(int step, int u, int j) const {
    const int k = step * S + DepthOf(u);
    // 16 bytes that reach past the end of their vector: those that end there,
    // moved down in Store.
    if constexpr (!kAcross) return data + (offset[u] + uint32_t(min(k * kScale + 16 * j, bytes * kScale - 16)));
    // Depth positions past the end read the last one and become zero in Store.
    return data + (uint32_t(min(k / kPosition + j, bytes / kPosition - 1)) * uint32_t(pitch) + offset[u]);
  }
  // kAnyByte: whether the fifth dword of a lane's 16 bytes is loaded. Of an 8-bit
  // row it mostly is the first one of the next lane's, whose 16 bytes follow in
  // memory: not at the end of a run of lanes, nor in the step that the depth ends
  // in, whose last granule is read from elsewhere than its place. (512 tiles of
  // 4097 bytes of depth: 16.9 us with every lane's loaded, 15.3 so. Across the
  // vectors a run is two lanes: 256 tiles 11.9 us, 15.1 so.)
  static constexpr bool kFifthFromNextLane = !kAcross && !kPlanes;
  __device__ __forceinline__ bool LoadsFifth(int step, int u) const {
    return !kFifthFromNextLane || (step + 1) * S > bytes || DepthOf(u) == S - 16;
  }
  __device__ __forceinline__ void Load(int step, Held& h) const {
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      if (!Exists(u)) continue;
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const char* from = From(step, u, j);
        if constexpr (!kAnyByte) {
          // (Runs start at multiples of 4 bytes, but the 16 bytes that end with one
          // do not where its length is no multiple. fp32 has no such.)
          if constexpr (kElement == 4)
            h.x[u][j] = *reinterpret_cast<const v4i_dwords*>(from);
          else
            h.x[u][j] = *reinterpret_cast<const granule::v4i_unaligned*>(from);
        } else {
          const int shift = static_cast<int>(reinterpret_cast<uintptr_t>(from) & 3);
          h.x[u][j] = *reinterpret_cast<const v4i_dwords*>(from - shift);
        }
      }
      if constexpr (kAnyByte) {
        if (LoadsFifth(step, u)) {
#pragma unroll
          for (int j = 0; j < kLoads; ++j) {
            const char* from = From(step, u, j);
            const int shift = static_cast<int>(reinterpret_cast<uintptr_t>(from) & 3);
            h.fifth[u][j] = *reinterpret_cast<const int*>(from - shift + (shift ? 16 : 12));
          }
        }
      }
    }
  }

  // Puts what Load has fetched of `step` into the slot. kInside: the step lies
  // inside the depth.
  template <bool kInside>
  __device__ __forceinline__ void Store(int step, const Held& h, char* slot) const {
    const bool partial = !kInside && (step + 1) * S > bytes;  // (wave-uniform)
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      if (!Exists(u)) continue;
      const int k = step * S + DepthOf(u);
      v4i x[kLoads];
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        x[j] = h.x[u][j];
        if constexpr (kAnyByte) {
          const uint32_t shift = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(From(step, u, j)) & 3);
          int fifth = h.fifth[u][j];
          if constexpr (kFifthFromNextLane) {
            // (row_shl:1: from the next lane of the 16.)
            const int next = __builtin_amdgcn_update_dpp(0, h.x[u][j][0], 0x101, 0xf, 0xf, false);
            if (!(partial || DepthOf(u) == S - 16)) fifth = next;
          }
#pragma unroll
          for (int d = 0; d < 4; ++d)
            x[j][d] = static_cast<int>(__builtin_amdgcn_alignbyte(d < 3 ? h.x[u][j][d + 1] : fifth, h.x[u][j][d], shift));
        }
        if constexpr (kAcross) {
          if (first + kTile > count)
            x[j] = PlaceGranule(x[j], (first * kScale + VectorOf(u)) * kColumnBytes, count * kScale * kColumnBytes);
        } else {
          if (partial) x[j] = PlaceGranule(x[j], k * kScale + 16 * j, bytes * kScale);
        }
      }
      const int vector = VectorOf(u);
      if constexpr (!kAcross && kPlanes) {
        // (Past the end: high 0, low -128, which meet zeros of the other operand.)
        v4i high, low;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const v4i& y = x[d / 2];
          high[d] = static_cast<int>(__builtin_amdgcn_perm(y[d % 2 * 2 + 1], y[d % 2 * 2], 0x07050301u));
          low[d] = static_cast<int>(__builtin_amdgcn_perm(y[d % 2 * 2 + 1], y[d % 2 * 2], 0x06040200u) ^ 0x80808080u);
        }
        *reinterpret_cast<v4i*>(slot + SlotOffset<S>(vector, DepthOf(u) / 16)) = high;
        *reinterpret_cast<v4i*>(slot + SlotOffset<S>(kTile + vector, DepthOf(u) / 16)) = low;
      } else if constexpr (!kAcross) {
        if constexpr (kElement == 1) {
          if (partial) {
#pragma unroll
            for (int d = 0; d < 4; ++d)  // (the padding stays zero)
              x[0][d] ^= static_cast<int>(flip & LowBytes(bytes - k - 4 * d));
          } else {
#pragma unroll
            for (int d = 0; d < 4; ++d) x[0][d] ^= static_cast<int>(flip);
          }
        }
        *reinterpret_cast<v4i*>(slot + SlotOffset<S>(vector, DepthOf(u) / 16)) = x[0];
      } else if constexpr (kElement == 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v4i y = {x[0][i], x[1][i], x[2][i], x[3][i]};
          if (partial) {
#pragma unroll
            for (int d = 0; d < 4; ++d) y[d] = k + 4 * d < bytes ? y[d] : 0;
          }
          *reinterpret_cast<v4i*>(slot + SlotOffset<S>(vector + i, DepthOf(u) / 16)) = y;
        }
      } else {
        const uint32_t valid = partial ? LowBytes(bytes - k) : 0xffffffffu;
#pragma unroll
        for (int quad = 0; quad < 4; ++quad) {
          // 4 x 4 bytes: t[i] = four depth positions of column 4 * quad + i.
          const uint32_t x0 = __builtin_amdgcn_perm(x[1][quad], x[0][quad], 0x05010400u);
          const uint32_t x1 = __builtin_amdgcn_perm(x[1][quad], x[0][quad], 0x07030602u);
          const uint32_t y0 = __builtin_amdgcn_perm(x[3][quad], x[2][quad], 0x05010400u);
          const uint32_t y1 = __builtin_amdgcn_perm(x[3][quad], x[2][quad], 0x07030602u);
          const uint32_t t[4] = {__builtin_amdgcn_perm(y0, x0, 0x05040100u), __builtin_amdgcn_perm(y0, x0, 0x07060302u),
                                 __builtin_amdgcn_perm(y1, x1, 0x05040100u), __builtin_amdgcn_perm(y1, x1, 0x07060302u)};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int column = vector + 4 * quad + i;
            const int to = kPlanes ? column / 2 + (i % 2 == 0 ? kTile : 0) : column;
            const uint32_t value = kPlanes ? (i % 2 == 0 ? t[i] ^ 0x80808080u : t[i]) : (t[i] ^ flip) & valid;
            *reinterpret_cast<uint32_t*>(slot + SlotOffset<S>(to, DepthOf(u) / 16) + DepthOf(u) % 16) = value;
          }
        }
      }
    }
  }
};

// LDS of a workgroup: the waves' slots, and later in the same memory their
// partial tiles (16 bytes - four consecutive rows of a column - at a time, in
// runs of 32 columns padded by one so that a column's pieces lie in different
// banks); behind that the partial sums of the tile's vectors and the
// write-back parameters of its rows and columns.
template <int kTile, int S, int kWaves, int kSlotVectors>
struct Memory {
  static constexpr int kVectors = 2 * kTile;
  static constexpr int kSlot = kSlotVectors * S;
  static constexpr int kBlocks = kTile / 32;              // 32 x 32 blocks each way
  static constexpr int kPart = kBlocks * kBlocks * 8 * 33;  // granules of a wave's partial tile
  static constexpr int kSums = std::max(kWaves * kSlot, kWaves * kPart * 16);
  static constexpr int kParams = kSums + kWaves * kVectors * 4;
  static constexpr int kBytes = kParams + 3 * kVectors * 4;
};

template <typename T, int kTile, int S, int kWaves, int kSourceA, int kSourceB>
__global__ __launch_bounds__(64 * kWaves, kWaves > 4 ? kWaves / 4 : 2) void SmallGemmKernel(GemmArgs args) {
  using SideA = Side<kTile, S, kSourceA, T::kElementA>;
  using SideB = Side<kTile, S, kSourceB, T::kElementB>;
  using Mem = Memory<kTile, S, kWaves, SideA::kSlotVectors + SideB::kSlotVectors>;
  constexpr int kBlocks = Mem::kBlocks;
  constexpr int kSubSteps = S / 32;
  extern __shared__ __attribute__((aligned(16))) char lds[];

  // The tile: every XCD (workgroups go to them round-robin) gets a contiguous
  // run of the tiles, in bands of four tile rows, so that those it holds share
  // operand panels in its L2.
  const int tiles_m = (args.M + kTile - 1) / kTile;
  const int tiles_n = (args.N + kTile - 1) / kTile;
  const int total = tiles_m * tiles_n;
  const int per_xcd = (total + 7) / 8;
  const int t = int(blockIdx.x % 8) * per_xcd + int(blockIdx.x / 8);
  if (t >= total) return;
  constexpr int kGroupM = 4;
  const int band = t / (kGroupM * tiles_n);
  const int band_rows = min(kGroupM, tiles_m - band * kGroupM);
  const int in_band = t - band * kGroupM * tiles_n;
  const int m0 = (band * kGroupM + in_band % band_rows) * kTile;
  const int n0 = in_band / band_rows * kTile;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = args.k_valid;  // depth in bytes
  const int steps = (K + S - 1) / S;
  const int my_steps = steps > wave ? (steps - wave + kWaves - 1) / kWaves : 0;

  SideA a;
  SideB b;
  a.Start(args.a, args.lda, args.M, m0, K, args.a_flip, lane);
  b.Start(args.b, args.ldb, args.N, n0, K, args.b_flip, lane);
  // Steps whose loads are in flight (16 waves: 128 registers a lane).
  constexpr int kAhead = kWaves > 8 ? 1 : 2;
  typename SideA::Held held_a[kAhead];
  typename SideB::Held held_b[kAhead];
  auto load = [&](int i, auto at) {
    a.Load(wave + kWaves * i, held_a[decltype(at)::value]);
    b.Load(wave + kWaves * i, held_b[decltype(at)::value]);
  };
  using First = std::integral_constant<int, 0>;
  using Second = std::integral_constant<int, kAhead - 1>;
  if (my_steps > 0) load(0, First());
  if (kAhead > 1 && my_steps > 1) load(1, Second());

  // What the write-back needs of the tile's rows and columns: fetched here,
  // a vector a thread, and used after the last step.
  typename T::Params params;
  const bool is_row = tid < kTile;
  if (tid < Mem::kVectors)
    T::LoadParams(args.ep, is_row, is_row ? min(m0 + tid, args.M - 1) : min(n0 + tid - kTile, args.N - 1), params);

  // (fp32: several accumulators in turn, so that the chains of additions are no
  // longer than where a depth is split over workgroups: four of eight waves, two
  // where there are more waves or the registers decide how many workgroups a CU
  // holds. Against 64 bits, 256 x 2048 x 256: split 2.1e-7, here 1.6e-7.)
  // (Two planes: an accumulator each.)
  constexpr bool kPlanes = SideA::kPlanes || SideB::kPlanes;
  constexpr bool kInteger = T::kElementA != 4;
  constexpr int kChains = kPlanes ? 2 : kInteger ? 1 : kWaves == 8 ? 4 : 2;
  static_assert(kBlocks == 1 || kChains == 1, "the larger tile exists for 8-bit operands");
  typename T::Acc acc[kBlocks][kBlocks][kChains];
  int sum_a[kBlocks], sum_b[kBlocks];
#pragma unroll
  for (int x = 0; x < kBlocks; ++x) {
    sum_a[x] = sum_b[x] = 0;
#pragma unroll
    for (int y = 0; y < kBlocks; ++y)
#pragma unroll
      for (int c = 0; c < kChains; ++c)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[x][y][c][v] = 0;
  }
  const bool sums_of_a = T::kElementA == 1 && args.fused_a_factor != 0;
  const bool sums_of_b = T::kElementB == 1 && args.fused_b_factor != 0;

  char* const slot = lds + wave * Mem::kSlot;
  // `steady`: a step that lies inside the depth and whose place step i + kAhead
  // takes. (Without conditions, or the wait for a step's loads is one for all
  // that may be in flight.)
  auto step_of = [&](int i, auto at, auto steady) {
    constexpr bool kSteady = decltype(steady)::value;
    const int step = wave + kWaves * i;
    a.template Store<kSteady>(step, held_a[decltype(at)::value], slot);
    b.template Store<kSteady>(step, held_b[decltype(at)::value], slot + SideA::kSlotVectors * S);
    if (kSteady || i + kAhead < my_steps) load(i + kAhead, at);
    // (Written and read by this wave only, whose LDS operations are performed
    // in order.)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    v4i fa[kSubSteps][kBlocks], fb[kSubSteps][kBlocks], low[kPlanes ? kSubSteps : 1];
#pragma unroll
    for (int ks = 0; ks < kSubSteps; ++ks) {
      // (32 vectors further on the swizzle is the same.)
      const int offset = SlotOffset<S>(lane & 31, ks * 2 + lane / 32);
#pragma unroll
      for (int x = 0; x < kBlocks; ++x) {
        fa[ks][x] = *reinterpret_cast<const v4i*>(slot + x * 32 * S + offset);
        fb[ks][x] = *reinterpret_cast<const v4i*>(slot + (SideA::kSlotVectors + x * 32) * S + offset);
      }
      if constexpr (kPlanes)
        low[ks] = *reinterpret_cast<const v4i*>(slot + (SideA::kPlanes ? kTile : SideA::kSlotVectors + kTile) * S + offset);
    }
#pragma unroll
    for (int ks = 0; ks < kSubSteps; ++ks) {
      if constexpr (kPlanes) {
        T::Mma(fa[ks][0], fb[ks][0], acc[0][0][0]);
        T::Mma(SideA::kPlanes ? low[ks] : fa[ks][0], SideB::kPlanes ? low[ks] : fb[ks][0], acc[0][0][1]);
      } else {
#pragma unroll
        for (int x = 0; x < kBlocks; ++x)
#pragma unroll
          for (int y = 0; y < kBlocks; ++y) T::Mma(fa[ks][x], fb[ks][y], acc[x][y], ks);
      }
    }
    if (sums_of_a) {
#pragma unroll
      for (int ks = 0; ks < kSubSteps; ++ks)
#pragma unroll
        for (int x = 0; x < kBlocks; ++x)
#pragma unroll
          for (int d = 0; d < 4; ++d) sum_a[x] = __builtin_amdgcn_sdot4(fa[ks][x][d], 0x01010101, sum_a[x], false);
    }
    if (sums_of_b) {
#pragma unroll
      for (int ks = 0; ks < kSubSteps; ++ks)
#pragma unroll
        for (int x = 0; x < kBlocks; ++x)
#pragma unroll
          for (int d = 0; d < 4; ++d) sum_b[x] = __builtin_amdgcn_sdot4(fb[ks][x][d], 0x01010101, sum_b[x], false);
    }
    __builtin_amdgcn_wave_barrier();
  };
  int i = 0;
  using Steady = std::true_type;
  using Last = std::false_type;
  if constexpr (kAhead == 1) {
    for (; i + 1 < my_steps; ++i) step_of(i, First(), Steady());
    if (i < my_steps) step_of(i, First(), Last());
  } else {
    for (; i + 3 < my_steps; i += 2) {
      step_of(i, First(), Steady());
      step_of(i + 1, Second(), Steady());
    }
    for (; i + 1 < my_steps; i += 2) {
      step_of(i, First(), Last());
      step_of(i + 1, Second(), Last());
    }
    if (i < my_steps) step_of(i, First(), Last());
  }

  // ---- the partial tiles, added through LDS ----
  __syncthreads();  // every wave is done with its slot
  v4i* const parts = reinterpret_cast<v4i*>(lds);
  int* const sums = reinterpret_cast<int*>(lds + Mem::kSums);
  int* const area = reinterpret_cast<int*>(lds + Mem::kParams);
  if (my_steps > 0) {
#pragma unroll
    for (int x = 0; x < kBlocks; ++x)
#pragma unroll
      for (int y = 0; y < kBlocks; ++y)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v4i w;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const auto& of = acc[x][y];
            typename T::Value sum = of[0][4 * q + e];
            if constexpr (kPlanes)
              sum = static_cast<int>(256u * static_cast<uint32_t>(sum) + static_cast<uint32_t>(of[1][4 * q + e]));
            if constexpr (kChains == 2 && !kPlanes) sum += of[1][4 * q + e];
            if constexpr (kChains == 4) sum = (sum + of[1][4 * q + e]) + (of[2][4 * q + e] + of[3][4 * q + e]);
            w[e] = T::Bits(sum);
          }
          // Rows 8 q + 4 (lane / 32) .. + 3 of column lane % 32 of the block.
          parts[wave * Mem::kPart + ((x * kBlocks + y) * 8 + 2 * q + lane / 32) * 33 + (lane & 31)] = w;
        }
    // Lanes l and l + 32 hold the two halves of a vector's sum.
    auto put = [&](int value, int vector) {
      const auto halves = __builtin_amdgcn_permlane32_swap(value, value, false, false);
      if (lane < 32) sums[wave * Mem::kVectors + vector + lane] = halves[0] + halves[1];
    };
#pragma unroll
    for (int x = 0; x < kBlocks; ++x) {
      if (sums_of_a) put(sum_a[x], x * 32);
      if (sums_of_b) put(sum_b[x], kTile + x * 32);
    }
  }
  if (tid < Mem::kVectors) T::StageParams(args.ep, is_row, params, area + tid, Mem::kVectors);
  __syncthreads();

  // A thread finishes four consecutive rows of a column. (A loop, not a lambda: in
  // one, captured, the kernel's arguments lie in memory for the compiler, and what a
  // lane chooses between two of them above becomes a load a lane from there, which
  // waits for all operand loads. 1024 x 1024 x 196 per channel: 5.5 us so, 5.0 with the loop.)
  const int active = min(steps, kWaves);
  constexpr int kQuads = kTile * kTile / 4;
#pragma unroll 1
  for (int quad = tid; quad < kQuads; quad += std::min(kQuads, 64 * kWaves)) {
    const int row = quad % (kTile / 4) * 4, col = quad / (kTile / 4);
    typename T::Value value[4] = {0, 0, 0, 0};
    uint32_t of_column = 0, of_row[4] = {0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w < active) {
        const v4i x = parts[w * Mem::kPart + ((row / 32 * kBlocks + col / 32) * 8 + row % 32 / 4) * 33 + col % 32];
#pragma unroll
        for (int e = 0; e < 4; ++e) value[e] += T::FromBits(x[e]);
        if (sums_of_a) {
          const v4i s = *reinterpret_cast<const v4i*>(sums + w * Mem::kVectors + row);
#pragma unroll
          for (int e = 0; e < 4; ++e) of_row[e] += static_cast<uint32_t>(s[e]);
        }
        if (sums_of_b) of_column += static_cast<uint32_t>(sums[w * Mem::kVectors + kTile + col]);
      }
    }
    if constexpr (kInteger) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        value[e] = static_cast<int>(static_cast<uint32_t>(value[e]) - static_cast<uint32_t>(args.fused_a_factor) * of_row[e] -
                                    static_cast<uint32_t>(args.fused_b_factor) * of_column);
    }
    int vals[4];
    T::Finish(value, area, Mem::kVectors, row, kTile + col, args.ep, vals);
    const int i0 = m0 + row, j = n0 + col;
    if (j >= args.N || i0 >= args.M) continue;
    char* const out = static_cast<char*>(args.dst.data) + (int64_t(j) * args.dst.cs + i0) * args.dst_elt;
    // (Stores of any width take any address.)
    if (i0 + 4 <= args.M) {
      if (args.dst_elt == 1) {
        const uint32_t w = uint32_t(vals[0] & 0xff) | uint32_t(vals[1] & 0xff) << 8 | uint32_t(vals[2] & 0xff) << 16 |
                           uint32_t(vals[3]) << 24;
        __builtin_memcpy(out, &w, sizeof(w));
      } else if (args.dst_elt == 2) {
        const uint32_t w[2] = {uint32_t(vals[0] & 0xffff) | uint32_t(vals[1]) << 16,
                               uint32_t(vals[2] & 0xffff) | uint32_t(vals[3]) << 16};
        __builtin_memcpy(out, w, sizeof(w));
      } else {
        __builtin_memcpy(out, vals, sizeof(vals));
      }
    } else {
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        if (i0 + e < args.M) {
          if (args.dst_elt == 1)
            reinterpret_cast<int8_t*>(out)[e] = static_cast<int8_t>(vals[e]);
          else if (args.dst_elt == 2)
            reinterpret_cast<int16_t*>(out)[e] = static_cast<int16_t>(vals[e]);
          else
            reinterpret_cast<int32_t*>(out)[e] = vals[e];
        }
      }
    }
  }
}

template <typename T, int kTile, int S, int kWaves, int kSourceA, int kSourceB>
hipError_t Launch(hipStream_t stream, const GemmArgs& args) {
  using Mem = Memory<kTile, S, kWaves,
                     Side<kTile, S, kSourceA, T::kElementA>::kSlotVectors + Side<kTile, S, kSourceB, T::kElementB>::kSlotVectors>;
  // (Rows: a granule must fit; across: 16 bytes of vectors.)
  if (args.k_valid < 16 || args.M < 16 || args.N < 16 || args.split_k != 1 || args.row_sums) return hipErrorInvalidValue;
  const int64_t total = int64_t((args.M + kTile - 1) / kTile) * ((args.N + kTile - 1) / kTile);
  if (total > (1 << 24)) return hipErrorInvalidValue;
  const int grid = static_cast<int>((total + 7) / 8 * 8);
  auto kernel = SmallGemmKernel<T, kTile, S, kWaves, kSourceA, kSourceB>;
  if (Mem::kBytes > 48 * 1024) {
    // Once per process and kernel; static initialisation is safe against concurrent callers.
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, Mem::kBytes);
    if (attr != hipSuccess) return attr;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * kWaves), Mem::kBytes, stream, args);
  return hipGetLastError();
}

// The forms on 32x32 tiles that the planners choose, and so the ones that are built.
template <typename T>
constexpr bool IsPlanned(int step, int waves, bool across, bool any_byte) {
  constexpr bool kPlanes = T::kElementA == 2 || T::kElementB == 2;
  constexpr bool kInt8 = T::kElementA == 1 && T::kElementB == 1;
  if (T::kElementA == 4 && any_byte) return false;
  if (step == 64) return waves == 4 || (waves == 8 && !(kInt8 && across));
  if (kPlanes || step != 128) return false;
  if (waves == 16) return !any_byte && (kInt8 || across);
  return across;
}

// The instantiation for a plan. Operands at any byte: both sides' byte forms
// (which read aligned ones as well).
template <typename T, int kTile, int S, int kWaves, int kSourceA, int kSourceB>
hipError_t LaunchPlanned(hipStream_t stream, const GemmArgs& args) {
  if constexpr (kTile == 64 || IsPlanned<T>(S, kWaves, IsAcross(kSourceA) || IsAcross(kSourceB), IsAnyByte(kSourceA)))
    return Launch<T, kTile, S, kWaves, kSourceA, kSourceB>(stream, args);
  return hipErrorInvalidValue;
}
template <typename T, int kTile, int S, int kWaves>
hipError_t LaunchSources(hipStream_t stream, const GemmArgs& args, const SmallGemmPlan& plan) {
  const bool across_a = IsAcross(plan.source_a), across_b = IsAcross(plan.source_b);
  if (IsAnyByte(plan.source_a) || IsAnyByte(plan.source_b)) {
    if (across_a && across_b) return LaunchPlanned<T, kTile, S, kWaves, kSmallAcrossBytes, kSmallAcrossBytes>(stream, args);
    if (across_a) return LaunchPlanned<T, kTile, S, kWaves, kSmallAcrossBytes, kSmallRowsBytes>(stream, args);
    if (across_b) return LaunchPlanned<T, kTile, S, kWaves, kSmallRowsBytes, kSmallAcrossBytes>(stream, args);
    return LaunchPlanned<T, kTile, S, kWaves, kSmallRowsBytes, kSmallRowsBytes>(stream, args);
  }
  if (across_a && across_b) return LaunchPlanned<T, kTile, S, kWaves, kSmallAcross, kSmallAcross>(stream, args);
  if (across_a) return LaunchPlanned<T, kTile, S, kWaves, kSmallAcross, kSmallRows>(stream, args);
  if (across_b) return LaunchPlanned<T, kTile, S, kWaves, kSmallRows, kSmallAcross>(stream, args);
  return LaunchPlanned<T, kTile, S, kWaves, kSmallRows, kSmallRows>(stream, args);
}
template <typename T>
hipError_t LaunchPlan(hipStream_t stream, const GemmArgs& args, const SmallGemmPlan& plan) {
  if (plan.tile == 64) {
    if constexpr (T::kElementA == 1 && T::kElementB == 1) {
      if (plan.step == 64 && plan.waves == 4) return LaunchSources<T, 64, 64, 4>(stream, args, plan);
      if (plan.step == 64 && plan.waves == 8) return LaunchSources<T, 64, 64, 8>(stream, args, plan);
    }
    return hipErrorInvalidValue;
  }
  if (plan.step == 64 && plan.waves == 4) return LaunchSources<T, 32, 64, 4>(stream, args, plan);
  if (plan.step == 64 && plan.waves == 8) return LaunchSources<T, 32, 64, 8>(stream, args, plan);
  if (plan.step == 128 && plan.waves == 4) return LaunchSources<T, 32, 128, 4>(stream, args, plan);
  if (plan.step == 128 && plan.waves == 8) return LaunchSources<T, 32, 128, 8>(stream, args, plan);
  if (plan.step == 128 && plan.waves == 16) return LaunchSources<T, 32, 128, 16>(stream, args, plan);
  return hipErrorInvalidValue;
}

}  // namespace small_gemm
}  // namespace ruyamd

#endif  // RUY_AMD_CSRC_KERNELS_SMALL_GEMM_H_
