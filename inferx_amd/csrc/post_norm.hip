// A branch's result that is normalised before it joins the residual stream, fused with the norm that follows:
//
//   d = delta / sqrt(mean(delta^2) + eps_d) * w_d;   h += d;   out = h / sqrt(mean(h^2) + eps) * w
//
// for layers that norm both before and after each branch.  One workgroup per row, everything in float32; h is
// float32 [T, width] and updated in place, unless `rows` picks rows out (then out[r] comes from row rows[r] and h
// stays).  With w null only the first two steps are done (nothing follows).
#include "common.h"

template <typename TD, typename TO>
__global__ void add_normed_rmsnorm_kernel(float* __restrict__ h, const TD* __restrict__ delta,
                                          const void* __restrict__ wd, int wd_dtype, float eps_d,
                                          const void* __restrict__ w, int w_dtype, float eps, TO* __restrict__ out,
                                          const int32_t* __restrict__ rows, int64_t width) {
  __shared__ float red[16];
  const int64_t r = blockIdx.x;
  const int64_t row = rows ? rows[r] : r;
  float* hr = h + row * width;
  const TD* dr = delta + row * width;
  float ssd = 0.f;
  for (int64_t i = threadIdx.x; i < width; i += blockDim.x) {
    const float d = ix_load(dr + i);
    ssd += d * d;
  }
  ssd = ix_block_sum(ssd, red);
  const float inv_d = 1.0f / sqrtf(ssd / static_cast<float>(width) + eps_d);
  float ss = 0.f;
  for (int64_t i = threadIdx.x; i < width; i += blockDim.x) {
    const float v = hr[i] + ix_load(dr + i) * inv_d * ix_load_rt(wd, wd_dtype, i);
    if (!rows) hr[i] = v;  // (read again below by the thread that wrote it)
    ss += v * v;
  }
  if (!w) return;
  ss = ix_block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / static_cast<float>(width) + eps);
  TO* outr = out + r * width;
  for (int64_t i = threadIdx.x; i < width; i += blockDim.x) {
    const float v = rows ? hr[i] + ix_load(dr + i) * inv_d * ix_load_rt(wd, wd_dtype, i) : hr[i];
    ix_store(outr + i, v * inv * ix_load_rt(w, w_dtype, i));
  }
}

// bfloat16 branch and output with a width that is a multiple of 4: NV times four columns per thread, which stay in
// registers, with everything that a row needs asked for at once (a column at a time, read again for each step: 2,048 rows of
// 2,048 17.9 us, now 11.8).
template <int NV>
__global__ void __launch_bounds__(1024)
add_normed_rmsnorm_vec4_kernel(float* __restrict__ h, const uint16_t* __restrict__ delta, const void* __restrict__ wd,
                               int wd_dtype, float eps_d, const void* __restrict__ w, int w_dtype, float eps,
                               uint16_t* __restrict__ out, const int32_t* __restrict__ rows, int64_t width) {
  __shared__ float red[16];
  const int64_t r = blockIdx.x;
  const int64_t row = rows ? rows[r] : r;
  float* hr = h + row * width;
  const uint16_t* dr = delta + row * width;
  float4 v[NV], d[NV], gd[NV], g[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) {  // (columns past the end: the first ones, not used)
    const int64_t c = 4 * (threadIdx.x + u * static_cast<int64_t>(blockDim.x)), at = c < width ? c : 0;
    d[u] = ix_load4_rt(dr, IX_BF16, at);
    v[u] = *reinterpret_cast<const float4*>(hr + at);
    gd[u] = ix_load4_rt(wd, wd_dtype, at);
    if (w) g[u] = ix_load4_rt(w, w_dtype, at);
  }
  auto squares = [&](const float4 (&x)[NV]) {
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < NV; ++u)
      if (4 * (threadIdx.x + u * static_cast<int64_t>(blockDim.x)) < width)
        ss += x[u].x * x[u].x + x[u].y * x[u].y + x[u].z * x[u].z + x[u].w * x[u].w;
    return ss;
  };
  const float inv_d = 1.0f / sqrtf(ix_block_sum(squares(d), red) / static_cast<float>(width) + eps_d);
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int64_t c = 4 * (threadIdx.x + u * static_cast<int64_t>(blockDim.x));
    v[u].x += d[u].x * inv_d * gd[u].x;
    v[u].y += d[u].y * inv_d * gd[u].y;
    v[u].z += d[u].z * inv_d * gd[u].z;
    v[u].w += d[u].w * inv_d * gd[u].w;
    if (!rows && c < width) *reinterpret_cast<float4*>(hr + c) = v[u];
  }
  if (!w) return;
  const float inv = 1.0f / sqrtf(ix_block_sum(squares(v), red) / static_cast<float>(width) + eps);
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int64_t c = 4 * (threadIdx.x + u * static_cast<int64_t>(blockDim.x));
    if (c < width)
      *reinterpret_cast<uint2*>(out + r * width + c) =
          ix_pack4_bf16(make_float4(v[u].x * inv * g[u].x, v[u].y * inv * g[u].y, v[u].z * inv * g[u].z, v[u].w * inv * g[u].w));
  }
}

extern "C" int ix_add_normed_rmsnorm(void* h, const void* delta, int delta_dtype, const void* wd, int wd_dtype,
                                     float eps_d, const void* w, int w_dtype, float eps, void* out, int out_dtype,
                                     const int32_t* rows, int64_t n_out_rows, int64_t width, hipStream_t stream) {
  IX_REQUIRE(width > 0 && n_out_rows >= 0, "sizes must be positive");
  IX_REQUIRE(delta != nullptr && wd != nullptr, "the branch's result and its norm's weight are needed");
  IX_REQUIRE((w == nullptr) == (out == nullptr), "a following norm and its output come together");
  if (n_out_rows == 0) return 0;
  dim3 grid(n_out_rows), block(width >= 4096 ? 1024 : (width >= 1024 ? 512 : 256));
  if (delta_dtype == IX_BF16 && (out == nullptr || out_dtype == IX_BF16) && width % 4 == 0 && width <= 8192 &&
      ((reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(delta) | reinterpret_cast<uintptr_t>(out)) & 15) == 0) {
#define VEC4(NV, THREADS)                                                                                             \
  hipLaunchKernelGGL(add_normed_rmsnorm_vec4_kernel<NV>, grid, dim3(THREADS), 0, stream, (float*)h, (const uint16_t*)delta, \
                     wd, wd_dtype, eps_d, w, w_dtype, eps, (uint16_t*)out, rows, width)
    if (width <= 1024) VEC4(1, 256);
    else if (width <= 2048) VEC4(1, 512);
    else if (width <= 4096) VEC4(2, 512);
    else VEC4(2, 1024);
#undef VEC4
    return ix_check_launch("ix_add_normed_rmsnorm");
  }
#define LAUNCH(TD, TO)                                                                                             \
  hipLaunchKernelGGL((add_normed_rmsnorm_kernel<TD, TO>), grid, block, 0, stream, (float*)h, (const TD*)delta, wd, \
                     wd_dtype, eps_d, w, w_dtype, eps, (TO*)out, rows, width)
  if (delta_dtype == IX_F32 && out_dtype == IX_F32) LAUNCH(float, float);
  else if (delta_dtype == IX_F32 && out_dtype == IX_BF16) LAUNCH(float, bf16_t);
  else if (delta_dtype == IX_BF16 && out_dtype == IX_F32) LAUNCH(bf16_t, float);
  else if (delta_dtype == IX_BF16 && out_dtype == IX_BF16) LAUNCH(bf16_t, bf16_t);
  else IX_REQUIRE(false, "dtypes must be float32 or bfloat16");
#undef LAUNCH
  return ix_check_launch("ix_add_normed_rmsnorm");
}
