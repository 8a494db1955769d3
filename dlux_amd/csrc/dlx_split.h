// Split of FP32 values into two bf16, the operand form of the split-BF16x3
// contractions: x = hi + lo + O(2^-17 |x|), all four products of the pairs.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dlx {

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_split_t;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2_split_t;

// Two floats -> two bf16 rounded to nearest even, packed (x0 in the low half):
// one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t bf16x2_rne(float x0, float x1) {
  const f32x2_split_t v = {x0, x1};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_split_t));
}

// Split of two values: x_i = hi_i + lo_i + O(2^-17 |x_i|), each pair packed.
// The residual is formed from the rounded x_i: contraction is off, so a
// product feeding x_i is never fused into the subtraction, and every producer
// of the same values writes the same bits whatever the code around it.
__device__ __forceinline__ void split2_bf16(float x0, float x1, uint32_t& hi, uint32_t& lo) {
#pragma clang fp contract(off)
  hi = bf16x2_rne(x0, x1);
  lo = bf16x2_rne(x0 - __uint_as_float(hi << 16), x1 - __uint_as_float(hi & 0xFFFF0000u));
}

}  // namespace dlx
