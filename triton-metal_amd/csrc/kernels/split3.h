/* fp32 values as three bf16 parts, x = hi + mid + lo, each the rounding of what
 * is left (24 bits in all): the operands of fp32 products on the bf16 MFMAs
 * (gemm_x3.hip, attn_x3.hip).  A product is the sum of the six of order 2^-16 and
 * above, small ones first; the three dropped are below 2^-26 of it. */
#ifndef TM_SPLIT3_H
#define TM_SPLIT3_H

#include "common.h"

/* two floats -> their bf16 roundings in one word, and what the roundings leave */
TM_DEV uint32_t x3_part(float &a, float &b) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef bf16_t b2 __attribute__((ext_vector_type(2)));
  const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, b2));
  a -= __uint_as_float(w << 16);
  b -= __uint_as_float(w & 0xffff0000u);
  return w;
}

/* the three parts of eight floats, each one MFMA operand's 16 bytes */
TM_DEV void x3_split8(float (&x)[8], u32x4 (&part)[3]) {
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[q][e] = x3_part(x[2 * e], x[2 * e + 1]);
}

/* Values are split 2^16 times as large, so that the lowest bit of every fp32
 * number, 2^-149, is one of bf16's, 2^-133 (the MFMAs and conversions keep
 * subnormals); results come out 2^32 (2^48: a product of a product) times as large.
 * What then leaves fp32's range -- a value from 2^112, a result from 2^96 (2^80) --
 * shows as a non-finite result, as do infinities and NaN, and is computed in fp32
 * instead. */
constexpr float X3_SCALE = 0x1p16f;
TM_DEV bool x3_not_finite(float x) { return !(x - x == 0.f); }

/* two products side by side: a product's six MFMAs wait for each other */
TM_DEV void mfma_x3_pair(const u32x4 (&a0)[3], const u32x4 (&b0)[3], f32x4 &c0, const u32x4 (&a1)[3],
                         const u32x4 (&b1)[3], f32x4 &c1) {
#pragma unroll
  for (int order = 2; order >= 0; --order)
#pragma unroll
    for (int q = order; q >= 0; --q) {
      c0 = mfma_16x16x32(__builtin_bit_cast(bf16x8, a0[q]), __builtin_bit_cast(bf16x8, b0[order - q]), c0);
      c1 = mfma_16x16x32(__builtin_bit_cast(bf16x8, a1[q]), __builtin_bit_cast(bf16x8, b1[order - q]), c1);
    }
}

#endif
