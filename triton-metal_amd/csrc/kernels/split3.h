/* fp32 values as three bf16 parts, x = hi + mid + lo, each the rounding of what
 * is left (24 bits in all): the operands of fp32 products on the bf16 MFMAs
 * (gemm_x3.hip, attn_x3.hip).  A product is the sum of eight of its nine partial
 * products, lo lo being below 2^-33 of it: hi hi in one accumulator, the seven
 * small ones in another, so that a result is rounded at its own magnitude once per
 * 32 products and a single product within 0.51 of its last place.  (With the six
 * of order 2^-16 and above in one accumulator a lone product was up to 0.94 of it
 * off.) */
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

/* hi[i], lo[i] += a[i] b[i], N products side by side: one product's seven small
 * MFMAs wait for each other */
template <int N>
TM_DEV void mfma_x3(const u32x4 (*const (&a)[N])[3], const u32x4 (*const (&b)[N])[3], f32x4 *const (&hi)[N],
                    f32x4 *const (&lo)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
    *hi[i] = mfma_16x16x32(__builtin_bit_cast(bf16x8, (*a[i])[0]), __builtin_bit_cast(bf16x8, (*b[i])[0]), *hi[i]);
#pragma unroll
  for (int order = 1; order <= 3; ++order)
#pragma unroll
    for (int q = order < 3 ? 0 : 1; q <= order && q < 3; ++q)
#pragma unroll
      for (int i = 0; i < N; ++i)
        *lo[i] = mfma_16x16x32(__builtin_bit_cast(bf16x8, (*a[i])[q]),
                               __builtin_bit_cast(bf16x8, (*b[i])[order - q]), *lo[i]);
}

#endif
