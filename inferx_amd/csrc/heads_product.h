// A wavefront's unit of the products that every head has of its own, for few rows (heads_product.hip says what bounds them): sixteen
// rows of a head's weights over the whole reduction, the first operand of v_mfma_f32_16x16x32_bf16, the tokens the columns.
#pragma once

#include "common.h"

typedef __bf16 hp_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 hp_bf16x4 __attribute__((ext_vector_type(4)));
typedef float hp_f32x4 __attribute__((ext_vector_type(4)));

// STEPS: pieces of 32 of the reduction that are on their way together
template <int STEPS>
__device__ __forceinline__ void hp_unit(const __bf16* __restrict__ x, int64_t x_t, int64_t x_h, const __bf16* __restrict__ w,
                                        __bf16* __restrict__ out, int64_t out_t, int64_t out_h, int tokens, int n, int width,
                                        int64_t unit) {
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const int per_head = n / 16;
  const int head = static_cast<int>(unit / per_head), row0 = 16 * static_cast<int>(unit % per_head);
  const __bf16* wr = w + (static_cast<int64_t>(head) * n + row0 + m) * width;
  const __bf16* xr = x + min(m, tokens - 1) * x_t + head * x_h;  // (columns past the last token: that one, not stored)
  hp_f32x4 acc = hp_f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < width; k0 += 32 * STEPS) {
    hp_bf16x8 wv[STEPS], xv[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int k = min(k0 + 32 * s, width - 32) + 8 * g;
      wv[s] = *reinterpret_cast<const hp_bf16x8*>(wr + k);
      xv[s] = *reinterpret_cast<const hp_bf16x8*>(xr + k);
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
      if (k0 + 32 * s < width) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[s], xv[s], acc, 0, 0, 0);
  }
  // lane holds weight rows row0 + 4 g + i of token m
  if (m < tokens)
    *reinterpret_cast<hp_bf16x4*>(out + m * out_t + head * out_h + row0 + 4 * g) =
        hp_bf16x4{(__bf16)acc[0], (__bf16)acc[1], (__bf16)acc[2], (__bf16)acc[3]};
}
