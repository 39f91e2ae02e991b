// Operand types of the 16-bit matrix instructions and the splits of an fp32 value into three bf16 or two fp16 pieces, shared by
// the kernels that run fp32 products on them (linear.hip, node_glue.hip).
#pragma once

#include "common.hpp"

namespace cm {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// a = hi + mid + lo with bf16 pieces (round to nearest at every step; the remainders are exact in fp32).  Two values at a
// time: the packed conversion rounds both and leaves the pieces in the order the matrix instruction takes them, and a
// piece widens back to fp32 by a shift or a mask (11 instructions per pair; element by element the compiler converts
// every value alone, widens it, and packs the pairs at the end with further conversions: 15).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split3_pair(float v0, float v1, unsigned &hi, unsigned &mid, unsigned &lo) {
  hi = __builtin_bit_cast(unsigned, __builtin_convertvector(f2{v0, v1}, bf16x2));
  const float r0 = v0 - __builtin_bit_cast(float, hi << 16), r1 = v1 - __builtin_bit_cast(float, hi & 0xffff0000u);
  mid = __builtin_bit_cast(unsigned, __builtin_convertvector(f2{r0, r1}, bf16x2));
  const float q0 = r0 - __builtin_bit_cast(float, mid << 16), q1 = r1 - __builtin_bit_cast(float, mid & 0xffff0000u);
  lo = __builtin_bit_cast(unsigned, __builtin_convertvector(f2{q0, q1}, bf16x2));
}
__device__ __forceinline__ void split3(f4 v, bf16x4 &hi, bf16x4 &mid, bf16x4 &lo) {
  unsigned h0, m0, l0, h1, m1, l1;
  split3_pair(v.x, v.y, h0, m0, l0);
  split3_pair(v.z, v.w, h1, m1, l1);
  hi = __builtin_bit_cast(bf16x4, u2{h0, h1});
  mid = __builtin_bit_cast(bf16x4, u2{m0, m1});
  lo = __builtin_bit_cast(bf16x4, u2{l0, l1});
}

// The split into two fp16 pieces, for v_mfma_f32_32x32x16_f16 and its like: s v = hi + lo with s a power of two that brings
// the largest value of the row (of X) or column (of W) that v belongs to to [2^14, 2^15).  Both pieces are rounded to nearest, so hi
// + lo is within 2^-24 of s v wherever |s v| >= 2^-1, i.e. down to 2^-15 of the row's largest value, and below that within 2^-25, 2^-39
// of the row's largest value.  Three piece products (hi hi, hi lo, lo hi) make the product; the dropped one, lo lo, is below 2^-24 of it.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split2_pair(float v0, float v1, float s, f16x2 &hi, f16x2 &lo) {
  const float a = v0 * s, b = v1 * s;
  hi = __builtin_convertvector(f2{a, b}, f16x2);
  lo = __builtin_convertvector(f2{a - static_cast<float>(hi.x), b - static_cast<float>(hi.y)}, f16x2);
}
__device__ __forceinline__ void split2(f4 v, float s, f16x4 &hi, f16x4 &lo) {
  f16x2 h0, l0, h1, l1;
  split2_pair(v.x, v.y, s, h0, l0);
  split2_pair(v.z, v.w, s, h1, l1);
  hi = __builtin_shufflevector(h0, h1, 0, 1, 2, 3);
  lo = __builtin_shufflevector(l0, l1, 0, 1, 2, 3);
}
// Scale of a row or column from its largest magnitude, and what takes it back: s = 2^-exponent.  `least`: the smallest biased
// exponent told apart (a smaller largest value, zero among them, is scaled as that one); infinities and NaN take the largest scale down.
struct PieceScale {
  float s;
  int exponent;
};
__device__ __forceinline__ PieceScale piece_scale(float largest, int least) {
  const int e = min(max(static_cast<int>(__float_as_uint(largest) >> 23), least), 254);
  return {__uint_as_float(static_cast<unsigned>(268 - e) << 23), e - 141};
}
constexpr int kLeastRowExponent = 14;     // s up to 2^127
constexpr int kLeastColumnExponent = 24;  // s up to 2^117: its inverse times the call's scale stays a normal number

}  // namespace cm
