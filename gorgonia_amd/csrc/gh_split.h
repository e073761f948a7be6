// float32 contractions on the bf16 matrix instructions.
//
// A float32 has 24 significant bits, a bf16 eight and the same exponents: x = h + m + l with three bf16 numbers, exactly
// (h is x rounded to nearest, m what is left rounded to nearest, l the rest).  Of the nine products of two such sums all but
// a.l b.l are added up, each exact in the multiplier; that one is at most 2^-34 of the product (|m| <= 2^-8 |x|, |l| <= 2^-17 |x|).
// (Without a.m b.l and a.l b.m as well, 2^-25 of the product each, a result of one product was off by up to 0.96 of its last
// place.)  The sums are float32, as on the float32 instructions, rounded once per instruction.  The seven products behind
// a.h b.h, at most 2^-7 of it together, have sums of their own: the large sum is rounded once per 16 k, and a result of one
// product (a diagonal, a scaling, a sparse row) is off by at most 0.51 of its last place, 0.5 on the float32 instructions.
// Eight instructions of 16 k take 130 ns on a SIMD where the eight float32 ones of 2 k take 217.
//
// Range: the inputs are scaled by 2^16, so that every bit of the smallest denormal stays inside bf16's (denormal) range
// and the split is exact for all inputs below 2^112; results are scaled back.  Larger, infinite and NaN inputs, and
// sums above 2^96, come out as an infinity or a NaN: a kernel tests what it summed and computes such a tile again with the
// float32 instructions.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

namespace gh_split {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kUp = 65536.0f;                          // of each operand
constexpr float kDown = 1.0f / (65536.0f * 65536.0f);   // of a product

// f(0), f(1), ... f(N - 1), each with its number as a constant
template <class F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void each(F&& f) { each_of(f, std::make_integer_sequence<int, (N > 0 ? N : 0)>{}); }

// Two values to their parts, a part of both in one register, in eight stages of one or two vector instructions.  An
// instruction that waits for the one before it costs a wavefront eight cycles; so the stages of a pair go behind one
// matrix instruction each, next to other stages of other pairs.
struct Pair {
  f32x2 rest, top;
  uint32_t part[3];
  template <int STAGE>
  __device__ __forceinline__ void stage(float x0, float x1) {
    if constexpr (STAGE == 0) rest = f32x2{x0 * kUp, x1 * kUp};
    if constexpr (STAGE == 1 || STAGE == 4 || STAGE == 7) part[STAGE / 3] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, bf16x2));
    if constexpr (STAGE == 2 || STAGE == 5) top = f32x2{__builtin_bit_cast(float, part[STAGE / 3] << 16), __builtin_bit_cast(float, part[STAGE / 3] & 0xffff0000u)};
    if constexpr (STAGE == 3 || STAGE == 6) { rest[0] -= top[0]; rest[1] -= top[1]; }
  }
};
constexpr int kStages = 8;

__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace gh_split
