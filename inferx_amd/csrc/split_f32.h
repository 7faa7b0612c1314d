// Float32 products on the bfloat16 matrix cores.
//
// A float32 number is the sum of three bfloat16 numbers of its sign: h, its upper sixteen bits, m, those of what is left, and l, what
// is left then: 3 x 8 bits are the 24 of float32, and every difference is exact.  Of the nine products of two such sums six are
// formed, h h, h m, m h, m m, h l and l h; m l, l m and l l are together below 2^-22 of the product, 2^-25 on average.  Each is exact in
// 32 bits, and sums are taken in 32 bits: h h in one accumulator, the five small ones, 2^-7 and less of it, in another, and
// both are added in the end.  So the large sums are rounded once for sixteen numbers of the reduction, where the float32 instruction
// (16 x 16 x 4) rounds them once for four.
//
// An infinity or a NaN makes its results no numbers (inf - inf); such results are formed again, one product after the other
// (`plain_dot`), so that they are what float32 gives.
#pragma once

#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Eight numbers' parts h, m, l.  (The empty assembly keeps the compiler from taking them for four whole numbers each, of which it then
// makes memory.)
__device__ __forceinline__ void split8(const f32x4& a, const f32x4& b, bf16x8 (&parts)[3]) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const auto upper = [](float lo, float hi) {  // the upper halves of two numbers, side by side
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
  };
  const auto rest = [](float v) { return v - __uint_as_float(__float_as_uint(v) & 0xffff0000u); };
  u32x4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = i < 2 ? a[2 * i] : b[2 * i - 4], y = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
    const float x1 = rest(x), y1 = rest(y);
    h[i] = upper(x, y);
    m[i] = upper(x1, y1);
    l[i] = upper(rest(x1), rest(y1));
  }
  bf16x8 p[3] = {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    asm("" : "+v"(p[i]));
    parts[i] = p[i];
  }
}

// The sum of n products in their order.
__device__ __attribute__((noinline)) float plain_dot(const float* x, const float* w, int n) {
  float sum = 0.f;
  for (int i = 0; i < n; ++i) sum = __builtin_fmaf(x[i], w[i], sum);
  return sum;
}
// (not an infinity, not a NaN)
__device__ __forceinline__ bool is_number(float v) { return fabsf(v) <= 3.4028234663852886e38f; }
