// A product of its own for every head, for few rows (decoding): out[t, h, :] = w[h] . x[t, h, :], bfloat16 operands, float32
// sums; w [heads, n, width], rows of x and out with strides of their own per token and head.  At most 16 tokens.
//
// What bounds it: the launch and one trip to memory (16 heads of 512 x 128: 2 MB of weights).  A wavefront takes sixteen rows
// of a head's weights over the whole reduction, as the first operand of v_mfma_f32_16x16x32_bf16, the tokens are the
// columns; up to 512 numbers of the reduction are asked for at once, and with few wavefronts each is a workgroup of its own.
// Eight tokens, 16 heads of 512 x 128 | 128 x 512: 3.2 | 3.7 us against 5.0 | 10.6 of the library's batched product.
#include "heads_product.h"

template <int STEPS>
__global__ void __launch_bounds__(256)
heads_product_kernel(const __bf16* __restrict__ x, int64_t x_t, int64_t x_h, const __bf16* __restrict__ w,
                     __bf16* __restrict__ out, int64_t out_t, int64_t out_h, int tokens, int heads, int n, int width) {
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (unit >= static_cast<int64_t>(heads) * (n / 16)) return;
  hp_unit<STEPS>(x, x_t, x_h, w, out, out_t, out_h, tokens, n, width, unit);
}

extern "C" int ix_heads_product(const void* x, int64_t x_t, int64_t x_h, const void* w, void* out, int64_t out_t, int64_t out_h,
                                int tokens, int heads, int n, int width, hipStream_t stream) {
  IX_REQUIRE(tokens > 0 && tokens <= 16 && heads > 0 && n > 0 && width > 0, "between 1 and 16 tokens, positive sizes");
  IX_REQUIRE(n % 16 == 0 && width % 32 == 0, "rows of weights in multiples of 16, the reduction in multiples of 32");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) == 0 && (x_t | x_h) % 8 == 0,
             "operands must lie on 16-byte boundaries");
  IX_REQUIRE((reinterpret_cast<uintptr_t>(out) & 7) == 0 && (out_t | out_h) % 4 == 0, "out must lie on 8-byte boundaries");
  const int64_t units = static_cast<int64_t>(heads) * (n / 16);
  IX_REQUIRE(units < (int64_t(1) << 31), "too many rows of weights for one launch");
  const unsigned per_group = units < 1024 ? 1 : 4;
  const dim3 grid(static_cast<unsigned>((units + per_group - 1) / per_group));
#define LAUNCH(STEPS)                                                                                                        \
  hipLaunchKernelGGL(heads_product_kernel<STEPS>, grid, dim3(64 * per_group), 0, stream, (const __bf16*)x, x_t, x_h,          \
                     (const __bf16*)w, (__bf16*)out, out_t, out_h, tokens, heads, n, width)
  if (width <= 128) LAUNCH(4);
  else LAUNCH(16);
#undef LAUNCH
  return ix_check_launch("ix_heads_product");
}
