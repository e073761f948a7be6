// float32 contractions on the bf16 matrix instructions.
//
// A float32 has 24 significant bits, a bf16 eight and the same exponents: x = h + m + l with three bf16 numbers, exactly
// (h is x rounded to nearest, m what is left rounded to nearest, l the rest).  Of the nine products of two such sums six are
// added up, a.h b.h, a.h b.m, a.m b.h, a.m b.m, a.h b.l and a.l b.h; each is exact in the multiplier.  The other three are
// at most 2^-25 of the product (a.m <= 2^-8 a, b.l <= 2^-17 b), half of what rounding the product to float32 may cost.
// The sums are float32, as on the float32 instructions, rounded to nearest once per instruction.  Six
// instructions of 16 k take 98 ns on a SIMD where the eight float32 ones of 2 k take 217.
//
// Range: the inputs are scaled by 2^16, so that every bit of the smallest denormal stays inside bf16's (denormal) range
// and the split is exact for all inputs below 2^112; results are scaled back.  Larger, infinite and NaN inputs, and
// sums above 2^96, come out as an infinity or a NaN: a kernel tests what it summed (split_finite) and computes such a tile
// again with the float32 instructions.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

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

// two values to their three parts, each part of the two in one register
__device__ __forceinline__ void pair(float x0, float x1, uint32_t* h, uint32_t* m, uint32_t* l) {
  f32x2 r = {x0 * kUp, x1 * kUp};
  uint32_t* const out[3] = {h, m, l};
#pragma unroll
  for (int p = 0; p < 3; p++) {
    const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
    *out[p] = u;
    r[0] -= __builtin_bit_cast(float, u << 16);
    r[1] -= __builtin_bit_cast(float, u & 0xffff0000u);
  }
}

// eight values that follow each other in k: one operand register group per part
__device__ __forceinline__ void eight(const float* x, u32x4* h, u32x4* m, u32x4* l) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    uint32_t a, b, c;
    pair(x[2 * i], x[2 * i + 1], &a, &b, &c);
    (*h)[i] = a; (*m)[i] = b; (*l)[i] = c;
  }
}

__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace gh_split
