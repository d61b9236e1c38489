// fp32 products on the bf16 matrix instructions by the published method of
// splitting a float into a sum of bf16 values (G. Henry, P. T. P. Tang, A. Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019: three parts, six products). A float is the sum of three
// bf16 values, each the rest of the ones before it rounded to nearest (24 bits of
// mantissa are three times 8), and of the nine products of two such sums the six
// largest are formed, high * high down to the 2^-16 terms. What is left out is at most
// 2^-24 of a product, a fifth of that in the mean, and has no sign of its
// own: a product counts with the bits of both factors to about its own 24th, not
// with all 48. Every bf16 product is exact, sums are fp32 throughout, and an instruction
// adds 16 depth positions with one rounding where the fp32 instruction adds two;
// the five smaller products have accumulators of their own. Measured against 64
// bits (values in [-1, 1], one accumulator chain): depth 256 7.8e-8 (fp32
// instructions 2.9e-7), 1024 1.9e-7 (6.1e-7), 3072 3.1e-7 (9.8e-7).
//
// The fp32 matrix instruction does 256 operations a clock and CU, the bf16 one
// 4096: six of them are 2.7 times as fast. The 5.5 vector instructions that
// split an element cost half as much energy again as its matrix instructions
// (random data, where the power limit sets the clock: 340 TFLOP/s of fp32
// products without them, 225 with, fp32 instructions 150), so elements are
// split as few times as possible.
//
// Not every float is such a sum: infinities and NaN are not, nor what a bf16 part
// rounds to infinity, nor most of what lies under 2^-110, whose last bits are below
// the smallest bf16 value (2^-133). The first two leave an accumulator that is not
// finite. The last leaves a remainder that the third part does not hold as a whole:
// one with bits in the lower half of its word, which are collected (Lost) and decide
// exactly (6 million bit patterns, subnormal ones among them: no disagreement). In
// either case the work is done again with fp32 instructions. How large the value lost
// is beside its own vector's does not matter: what it meets in the other operand may
// be large, and what its neighbours meet zero.
//
// What that costs, us, ordinary values / such a value in the first steps of every wave,
// with which the loop ends / in the last / an infinity, which only the sums show (and
// fp32 instructions throughout, as before there were parts): 1024^3 19.7 / 26.8 / 34.0 /
// 33.9 (22.3), 1537 x 1111 x 2051 54.8 / 86.4 / 118.7 / 118.9 (72.5), 2048 x 3072 x 2048
// 139.5 / 204 / 324 / 325 (186), 512 x 4096 x 512 22.1 / 29.5 / 36.0 / 36.1 (23.0).
#ifndef RUY_AMD_CSRC_KERNELS_FLOAT_PARTS_H_
#define RUY_AMD_CSRC_KERNELS_FLOAT_PARTS_H_

#include <hip/hip_runtime.h>

#include "granule.h"

namespace ruyamd {
namespace float_parts {

using granule::v4i;
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// Two floats rounded to bf16 in one register, and its two halves as floats.
__device__ __forceinline__ int RoundPair(float x, float y) {
  const v2f both = {x, y};
  return __builtin_bit_cast(int, __builtin_convertvector(both, v2bf));
}
__device__ __forceinline__ float LowHalf(int pair) { return __int_as_float(pair << 16); }
__device__ __forceinline__ float HighHalf(int pair) { return __int_as_float(pair & static_cast<int>(0xffff0000u)); }

// Eight depth values of a vector: two granules of floats, as the operands of one
// matrix instruction a part. part[0] + part[1] + part[2] are the values.
struct Parts {
  v4i part[3];
};

// The splitting of one granule (four floats), an instruction or two at a time so
// that a schedule can deal them out between matrix instructions (which leave a
// wave five or six issue slots each). kSplitOps pieces: Op<0>() ... in order.
constexpr int kSplitOps = 22;
struct Splitter {
  float rest[4];
  int pair[2];
  // (dot2 instructions, which would subtract a half without extracting it,
  // wait for the matrix pipe: 22 cycles each behind a matrix instruction.)
  template <int kOp>
  __device__ __forceinline__ void Op(const v4i& x, int which, Parts& to, int& lost) {
    if constexpr (kOp < 20) {
      constexpr int part = kOp / 10, op = kOp % 10;
      if constexpr (op < 2) {
        if constexpr (part == 0) {
          rest[2 * op] = __int_as_float(x[2 * op]);
          rest[2 * op + 1] = __int_as_float(x[2 * op + 1]);
        }
        pair[op] = RoundPair(rest[2 * op], rest[2 * op + 1]);
        to.part[part][2 * which + op] = pair[op];
      } else {
        constexpr int e = (op - 2) % 4;
        if constexpr (op < 6)
          half[e] = e % 2 ? HighHalf(pair[e / 2]) : LowHalf(pair[e / 2]);
        else
          rest[e] -= half[e];
      }
    } else {
      constexpr int e = 2 * (kOp - 20);
      to.part[2][2 * which + kOp - 20] = RoundPair(rest[e], rest[e + 1]);
      // (As text, in place: the compiler collects the remainders in registers otherwise.)
      asm volatile("v_or3_b32 %0, %1, %2, %0" : "+v"(lost) : "v"(rest[e]), "v"(rest[e + 1]));
    }
  }
  float half[4];
};

// Product number e (0 .. 5) of two vectors' parts, the smallest first; the last
// one is high * high.
constexpr int kProducts = 6;
constexpr int kPartOfA[kProducts] = {2, 0, 1, 1, 0, 0};
constexpr int kPartOfB[kProducts] = {0, 2, 1, 0, 1, 0};
// (Given the builtin, the compiler moves the accumulators between the two
// register files on every trip round a loop. What the assembler text keeps from
// it: Drain() in front of the first ordinary read of the accumulators, which
// it names so that no copy of one can be made ahead of it. Nor does the compiler know
// of the two wait states that a matrix instruction needs behind a vector instruction
// that writes what it reads: Settle() brings them behind whatever clears or copies
// accumulators, in front of a loop and behind it. Both are places where it would be
// free to do either anyway; a test looks for it in the assembly of the whole kernel.)
template <int kProduct>
__device__ __forceinline__ void Mma(const Parts& a, const Parts& b, v16f& acc) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0"
               : "+a"(acc)
               : "v"(a.part[kPartOfA[kProduct]]), "v"(b.part[kPartOfB[kProduct]]));
}
// (To the compiler the accumulators are registers like any other from there on.
// Otherwise it clears others for the way past a loop and copies all of them behind
// it: 1024^3 0.4 us.)
template <int kA, int kB>
__device__ __forceinline__ void Settle(v16f (&x)[kA][kB], v16f (&y)[kA][kB]) {
#pragma unroll
  for (int b = 0; b < kA * kB; ++b) asm volatile("" : "+a"(x[b / kB][b % kB]), "+a"(y[b / kB][b % kB]));
  asm volatile("s_nop 1" : "+a"(x[0][0]), "+a"(y[0][0]));
}
template <int kA, int kB>
__device__ __forceinline__ void Drain(v16f (&x)[kA][kB], v16f (&y)[kA][kB]) {
  asm volatile("s_nop 15\n\ts_nop 7" : "+a"(x[0][0]), "+a"(y[0][0]));
#pragma unroll
  for (int b = 1; b < kA * kB; ++b) asm volatile("" : "+a"(x[b / kB][b % kB]), "+a"(y[b / kB][b % kB]));
}

// The OR of elements' last remainders: whether one of the elements is not the sum of
// its parts.
__device__ __forceinline__ bool Lost(int lost) { return (lost & 0xffff) != 0; }

}  // namespace float_parts
}  // namespace ruyamd

#endif  // RUY_AMD_CSRC_KERNELS_FLOAT_PARTS_H_
