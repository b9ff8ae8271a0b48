// fp32 values as three bf16 parts, for products with fp32 accuracy on the
// bf16 matrix cores. (Splitting a value into a sum of narrower ones for exact
// partial products goes back to T. J. Dekker, "A floating-point technique for
// extending the available precision", 1971.)
//
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m): 8
// significant bits each, the differences exact. Operands are split as 2^24 x:
// bf16 has the exponents of fp32 but ends at 2^-133, so below 2^-111 the third
// part of x itself, then the second, would be cut off (relative error 5e-5 at
// 2^-120). Scaled, the parts of any fp32 value are normal bf16 values (the
// matrix cores take subnormal ones, with fewer bits of the product). The
// factors are powers of two, so results come out with the same bits after
// their inverse (a product of two operands carries 2^48). It costs one vector
// instruction a value, 0 to 6 % of a kernel (MI355X, us: GEMMs of 2048 x 50304 x
// 768 960 -> 958, 2048 x 2304 x 768 55.0 -> 56.7, 2048 x 768 x 768 23.1 -> 24.4;
// flash dK and dV of 8 x 2048 x 16 x 64 822 -> 836). A product takes the six
// partial products of order 2^-16 and larger, hh + hm + mh + mm + hl + lh, on
// v_mfma_f32_32x32x16_bf16 with fp32 accumulation; what is left out is below
// 2^-25 of a product. Six of them do the work of eight v_mfma_f32_32x32x2_f32
// in 192 matrix-core cycles instead of 512 and round the accumulator 6 times
// per 16 k instead of 8. The parts of a value that is not finite, or that
// passes the largest finite one when scaled (from 2^104), hold a NaN or
// infinities of both signs, so its products come out as NaN: kernels take
// those results, and no others, from fp32 products.
#pragma once

#include "skv_common.h"

namespace skv {

typedef float split_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float split_f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ bool finite(float x) { return fabsf(x) <= 3.402823466e38f; }

constexpr float kSplitScale = 0x1p24f;    // of every operand
constexpr float kSplitUnscale = 0x1p-48f;  // of a product of two

// Two scaled values as three words of two parts each (the first in the low half).
// (No contraction: x is a rounded value, also where it is a product.)
__device__ __forceinline__ void split2(float x, float y, uint32_t& h, uint32_t& m, uint32_t& l) {
#pragma clang fp contract(off)
  h = __builtin_bit_cast(uint32_t, __builtin_convertvector(split_f32x2{x, y}, bf16x2));
  const float rx = x - bf16w_lo(h), ry = y - bf16w_hi(h);
  m = __builtin_bit_cast(uint32_t, __builtin_convertvector(split_f32x2{rx, ry}, bf16x2));
  l = __builtin_bit_cast(uint32_t,
                         __builtin_convertvector(
                             split_f32x2{rx - bf16w_lo(m), ry - bf16w_hi(m)}, bf16x2));
}

// The parts (planes 0 h, 1 m, 2 l) of the two factors in the six partial
// products, small ones first.
constexpr int kSplitA[6] = {2, 0, 1, 1, 0, 0}, kSplitB[6] = {0, 2, 1, 0, 1, 0};

// c += A B over 16 k.
__device__ __forceinline__ split_f32x16 mfma_split(const bf16x8 (&a)[3], const bf16x8 (&b)[3],
                                                   split_f32x16 c) {
#pragma unroll
  for (int t = 0; t < 6; ++t)
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kSplitA[t]], b[kSplitB[t]], c, 0, 0, 0);
  return c;
}

// hi += the leading partial product over 16 k, lo += the other five: a long
// sum kept as hi + lo rounds at its full magnitude once per 16 k instead of 6
// times.
__device__ __forceinline__ void mfma_split(const bf16x8 (&a)[3], const bf16x8 (&b)[3],
                                           split_f32x16& hi, split_f32x16& lo) {
#pragma unroll
  for (int t = 0; t < 5; ++t)
    lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kSplitA[t]], b[kSplitB[t]], lo, 0, 0, 0);
  hi = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], hi, 0, 0, 0);
}

}  // namespace skv
