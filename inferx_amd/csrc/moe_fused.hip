// The weighted sum of the routed experts' outputs, the shared expert, the
// residual add and the RMSNorm that follows, in one pass over a token's row:
//   v = h[row] + sum_s topk_w[row, s] * y[dest[row, s]] + gate[row] * shared[row]
//   h[row] = v (unless rows are picked);  out = v * rsqrt(mean(v^2) + eps) * w
// Arithmetic and order of additions are those of ix_moe_combine followed by
// ix_add_rmsnorm, except that the feed-forward's sum is not rounded to the
// activations' type before it joins the float32 residual stream.
// With `wd` the feed-forward's sum passes an RMS norm of its own first (layers that norm a branch's result as well):
//   f = sum ...;  v = h[row] + f * rsqrt(mean(f^2) + eps_d) * wd
#include "common.h"

template <typename T>
__global__ void moe_combine_add_rmsnorm_kernel(float* __restrict__ h, const T* __restrict__ y,
                                               const int32_t* __restrict__ dest, const float* __restrict__ topk_w,
                                               const T* __restrict__ shared, const float* __restrict__ shared_gate,
                                               const void* __restrict__ w, int w_dtype, T* __restrict__ out,
                                               const int32_t* __restrict__ rows, int64_t row_width, int64_t width,
                                               int k, float eps, const void* __restrict__ wd, int wd_dtype,
                                               float eps_d) {
  // (`width` is what one norm runs over: the row, or one of its gridDim.y equal runs, each with its own sum)
  extern __shared__ __align__(16) float vrow[];  // [width]
  __shared__ float red[16];
  __shared__ float sw[32];
  __shared__ int32_t sd[32];
  const int64_t r = blockIdx.x;
  const int64_t row = rows ? rows[r] : r;
  if (threadIdx.x < k) {
    sw[threadIdx.x] = topk_w[row * k + threadIdx.x];
    sd[threadIdx.x] = dest[row * k + threadIdx.x];
  }
  __syncthreads();
  const float sg = shared ? (shared_gate ? shared_gate[row] : 1.0f) : 0.f;
  const int64_t first = blockIdx.y * width;
  float* hr = h + row * row_width + first;
  y += first;
  if (shared) shared += first;
  float sumsq = 0.f;
  if (wd) {  // the sum is normalised before it is added
    float sumsq_d = 0.f;
    for (int64_t c = threadIdx.x; c < width; c += blockDim.x) {
      float acc = 0.f;
      for (int s = 0; s < k; ++s) acc += sw[s] * ix_load(y + static_cast<int64_t>(sd[s]) * row_width + c);
      if (shared) acc += sg * ix_load(shared + row * row_width + c);
      vrow[c] = acc;
      sumsq_d += acc * acc;
    }
    sumsq_d = ix_block_sum(sumsq_d, red);
    const float inv_d = 1.0f / sqrtf(sumsq_d / static_cast<float>(width) + eps_d);
    for (int64_t c = threadIdx.x; c < width; c += blockDim.x) {  // (every thread reads back what it wrote itself)
      const float v = hr[c] + vrow[c] * inv_d * ix_load_rt(wd, wd_dtype, first + c);
      if (!rows) hr[c] = v;
      vrow[c] = v;
      sumsq += v * v;
    }
  } else {
    for (int64_t c = threadIdx.x; c < width; c += blockDim.x) {
      float acc = 0.f;
      for (int s = 0; s < k; ++s) acc += sw[s] * ix_load(y + static_cast<int64_t>(sd[s]) * row_width + c);
      if (shared) acc += sg * ix_load(shared + row * row_width + c);
      const float v = hr[c] + acc;
      if (!rows) hr[c] = v;
      vrow[c] = v;
      sumsq += v * v;
    }
  }
  sumsq = ix_block_sum(sumsq, red);
  const float inv = 1.0f / sqrtf(sumsq / static_cast<float>(width) + eps);
  T* outr = out + r * row_width + first;
  for (int64_t c = threadIdx.x; c < width; c += blockDim.x) ix_store(outr + c, vrow[c] * inv * ix_load_rt(w, w_dtype, first + c));
}

// bfloat16 with a width that is a multiple of 4: four columns per thread (8-byte loads of the experts' rows,
// 16-byte ones of the residual stream); the same additions in the same order as above.
__device__ __forceinline__ void bf16x4_to_f32(uint2 p, float (&f)[4]) {
  f[0] = __uint_as_float(p.x << 16);
  f[1] = __uint_as_float(p.x & 0xffff0000u);
  f[2] = __uint_as_float(p.y << 16);
  f[3] = __uint_as_float(p.y & 0xffff0000u);
}

__global__ void moe_combine_add_rmsnorm_vec4_kernel(float* __restrict__ h, const uint16_t* __restrict__ y,
                                                    const int32_t* __restrict__ dest,
                                                    const float* __restrict__ topk_w,
                                                    const uint16_t* __restrict__ shared,
                                                    const float* __restrict__ shared_gate, const void* __restrict__ w,
                                                    int w_dtype, uint16_t* __restrict__ out,
                                                    const int32_t* __restrict__ rows, int64_t row_width, int64_t width,
                                                    int k, float eps, const void* __restrict__ wd, int wd_dtype,
                                                    float eps_d) {
  extern __shared__ __align__(16) float vrow[];  // [width]
  __shared__ float red[16];
  __shared__ float sw[32];
  __shared__ int32_t sd[32];
  const int64_t r = blockIdx.x;
  const int64_t row = rows ? rows[r] : r;
  if (threadIdx.x < k) {
    sw[threadIdx.x] = topk_w[row * k + threadIdx.x];
    sd[threadIdx.x] = dest[row * k + threadIdx.x];
  }
  __syncthreads();
  const float sg = shared ? (shared_gate ? shared_gate[row] : 1.0f) : 0.f;
  const int64_t first = blockIdx.y * width;
  float* hr = h + row * row_width + first;
  y += first;
  if (shared) shared += first;
  float sumsq = 0.f;
  float inv_d = 1.0f;
  if (wd) {  // the sum is normalised before it is added: its sum of squares first (the sum itself is formed twice)
    float sumsq_d = 0.f;
    for (int64_t c = 4 * threadIdx.x; c < width; c += 4 * blockDim.x) {
      float acc[4] = {0.f, 0.f, 0.f, 0.f}, f[4];
      for (int s = 0; s < k; ++s) {
        bf16x4_to_f32(*reinterpret_cast<const uint2*>(y + static_cast<int64_t>(sd[s]) * row_width + c), f);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += sw[s] * f[i];
      }
      if (shared) {
        bf16x4_to_f32(*reinterpret_cast<const uint2*>(shared + row * row_width + c), f);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += sg * f[i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sumsq_d += acc[i] * acc[i];
    }
    sumsq_d = ix_block_sum(sumsq_d, red);
    inv_d = 1.0f / sqrtf(sumsq_d / static_cast<float>(width) + eps_d);
  }
  for (int64_t c = 4 * threadIdx.x; c < width; c += 4 * blockDim.x) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, f[4];
    for (int s = 0; s < k; ++s) {
      bf16x4_to_f32(*reinterpret_cast<const uint2*>(y + static_cast<int64_t>(sd[s]) * row_width + c), f);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += sw[s] * f[i];
    }
    if (shared) {
      bf16x4_to_f32(*reinterpret_cast<const uint2*>(shared + row * row_width + c), f);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += sg * f[i];
    }
    if (wd) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] *= inv_d * ix_load_rt(wd, wd_dtype, first + c + i);
    }
    float4 v = *reinterpret_cast<const float4*>(hr + c);
    v.x += acc[0]; v.y += acc[1]; v.z += acc[2]; v.w += acc[3];
    if (!rows) *reinterpret_cast<float4*>(hr + c) = v;
    *reinterpret_cast<float4*>(vrow + c) = v;
    sumsq += v.x * v.x;
    sumsq += v.y * v.y;
    sumsq += v.z * v.z;
    sumsq += v.w * v.w;
  }
  sumsq = ix_block_sum(sumsq, red);
  const float inv = 1.0f / sqrtf(sumsq / static_cast<float>(width) + eps);
  uint16_t* outr = out + r * row_width + first;
  for (int64_t c = 4 * threadIdx.x; c < width; c += 4 * blockDim.x) {
    const float4 v = *reinterpret_cast<const float4*>(vrow + c);
    uint2 o;
    o.x = ix_f32_to_bf16(v.x * inv * ix_load_rt(w, w_dtype, first + c)) |
          static_cast<uint32_t>(ix_f32_to_bf16(v.y * inv * ix_load_rt(w, w_dtype, first + c + 1))) << 16;
    o.y = ix_f32_to_bf16(v.z * inv * ix_load_rt(w, w_dtype, first + c + 2)) |
          static_cast<uint32_t>(ix_f32_to_bf16(v.w * inv * ix_load_rt(w, w_dtype, first + c + 3))) << 16;
    *reinterpret_cast<uint2*>(outr + c) = o;
  }
}

// The same without a norm of the sum, NV times four columns per thread in registers: the stream, the shared expert's row and
// the weight are asked for while the row's places among the experts' are looked up, those eight at a time (one after the
// other, through LDS: 2,048 rows of 2,048 from four experts 20.4 us, now 16.1; eight rows 5.6, now 4.7).
#define CMB_SLOTS 8
template <int NV>
__global__ void __launch_bounds__(1024)
moe_combine_add_rmsnorm_rows_kernel(float* __restrict__ h, const uint16_t* __restrict__ y, const int32_t* __restrict__ dest,
                                    const float* __restrict__ topk_w, const uint16_t* __restrict__ shared,
                                    const float* __restrict__ shared_gate, const void* __restrict__ w, int w_dtype,
                                    uint16_t* __restrict__ out, const int32_t* __restrict__ rows, int64_t row_width,
                                    int64_t width, int k, float eps) {
  __shared__ float red[16];
  const int64_t r = blockIdx.x;
  const int64_t row = rows ? rows[r] : r;
  const int64_t first = blockIdx.y * width;
  float* hr = h + row * row_width + first;
  const uint16_t* sr = shared ? shared + row * row_width + first : nullptr;
  const uint16_t* yr = y + first;
  int64_t at[NV];
  float4 v[NV], g[NV];
  uint2 sh[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) {  // (columns past the end: the first ones, not used)
    const int64_t c = 4 * (threadIdx.x + u * static_cast<int64_t>(blockDim.x));
    at[u] = c < width ? c : 0;
    v[u] = *reinterpret_cast<const float4*>(hr + at[u]);
    sh[u] = sr ? *reinterpret_cast<const uint2*>(sr + at[u]) : make_uint2(0u, 0u);
    g[u] = ix_load4_rt(w, w_dtype, first + at[u]);
  }
  const float sg = shared ? (shared_gate ? shared_gate[row] : 1.0f) : 0.f;
  float acc[NV][4] = {};
  for (int s0 = 0; s0 < k; s0 += CMB_SLOTS) {
    uint2 part[CMB_SLOTS][NV];
    float sw[CMB_SLOTS];
#pragma unroll
    for (int s = 0; s < CMB_SLOTS; ++s) {
      if (s0 + s >= k) break;
      sw[s] = topk_w[row * k + s0 + s];
      const uint16_t* from = yr + static_cast<int64_t>(dest[row * k + s0 + s]) * row_width;
#pragma unroll
      for (int u = 0; u < NV; ++u) part[s][u] = *reinterpret_cast<const uint2*>(from + at[u]);
    }
#pragma unroll
    for (int s = 0; s < CMB_SLOTS; ++s) {
      if (s0 + s >= k) break;
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        float f[4];
        bf16x4_to_f32(part[s][u], f);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u][i] += sw[s] * f[i];
      }
    }
  }
  float sumsq = 0.f;
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    if (sr) {
      float f[4];
      bf16x4_to_f32(sh[u], f);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[u][i] += sg * f[i];
    }
    v[u].x += acc[u][0]; v[u].y += acc[u][1]; v[u].z += acc[u][2]; v[u].w += acc[u][3];
    if (4 * (threadIdx.x + u * static_cast<int64_t>(blockDim.x)) < width) sumsq = ix_add_squares(sumsq, v[u]);
  }
  sumsq = ix_block_sum(sumsq, red);
  const float inv = 1.0f / sqrtf(sumsq / static_cast<float>(width) + eps);
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int64_t c = 4 * (threadIdx.x + u * static_cast<int64_t>(blockDim.x));
    if (c >= width) continue;
    if (!rows) *reinterpret_cast<float4*>(hr + c) = v[u];
    *reinterpret_cast<uint2*>(out + r * row_width + first + c) =
        ix_pack4_bf16(make_float4(v[u].x * inv * g[u].x, v[u].y * inv * g[u].y, v[u].z * inv * g[u].z, v[u].w * inv * g[u].w));
  }
}

extern "C" int ix_moe_combine_add_rmsnorm(void* h, const void* y, int dtype, const int32_t* dest,
                                          const float* topk_w, const void* shared, const float* shared_gate,
                                          const void* w, int w_dtype, void* out, const int32_t* rows,
                                          int64_t n_out_rows, int64_t row_width, int k, float eps, const void* wd,
                                          int wd_dtype, float eps_d, int groups, hipStream_t stream) {
  // `groups`: the last norm runs over that many equal runs of the row, each with its own root mean square
  IX_REQUIRE(n_out_rows >= 0 && row_width > 0, "sizes must be positive");
  IX_REQUIRE(groups > 0 && groups <= 65535 && row_width % groups == 0, "the groups must divide the width");
  IX_REQUIRE(groups == 1 || wd == nullptr, "a sum with a norm of its own goes with a last norm in one group");
  const int64_t width = row_width / groups;
  IX_REQUIRE(k > 0 && k <= 32, "top_k must be between 1 and 32");
  IX_REQUIRE(width * sizeof(float) <= 60 * 1024, "hidden width too large for the fused kernel (limit 15360)");
  IX_REQUIRE(w_dtype == IX_F32 || w_dtype == IX_BF16, "weight dtype must be float32 or bfloat16");
  if (n_out_rows == 0) return 0;
  dim3 grid(n_out_rows, groups), block(width >= 4096 ? 1024 : (width >= 1024 ? 512 : 256));
  const size_t smem = width * sizeof(float);
  if (dtype == IX_F32)
    hipLaunchKernelGGL(moe_combine_add_rmsnorm_kernel<float>, grid, block, smem, stream, (float*)h, (const float*)y,
                       dest, topk_w, (const float*)shared, shared_gate, w, w_dtype, (float*)out, rows, row_width, width, k, eps,
                       wd, wd_dtype, eps_d);
  else if (dtype == IX_BF16 && width % 4 == 0 && wd == nullptr && width <= 8192 &&
           ((reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(shared) |
             reinterpret_cast<uintptr_t>(out)) & 15) == 0) {
#define ROWS(NV, THREADS)                                                                                             \
  hipLaunchKernelGGL(moe_combine_add_rmsnorm_rows_kernel<NV>, grid, dim3(THREADS), 0, stream, (float*)h, (const uint16_t*)y, \
                     dest, topk_w, (const uint16_t*)shared, shared_gate, w, w_dtype, (uint16_t*)out, rows, row_width, width, k, eps)
    if (width <= 1024) ROWS(1, 256);
    else if (width < 2048) ROWS(2, 256);
    else if (width == 2048) ROWS(1, 512);
    else if (width < 4096) ROWS(2, 512);
    else if (width == 4096) ROWS(1, 1024);
    else ROWS(2, 1024);
#undef ROWS
  } else if (dtype == IX_BF16 && width % 4 == 0 &&
           ((reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(shared) |
             reinterpret_cast<uintptr_t>(out)) & 15) == 0)
    hipLaunchKernelGGL(moe_combine_add_rmsnorm_vec4_kernel, grid, dim3(width >= 4096 ? 1024 : (width >= 2048 ? 512 : 256)),
                       smem, stream, (float*)h, (const uint16_t*)y, dest, topk_w, (const uint16_t*)shared, shared_gate, w,
                       w_dtype, (uint16_t*)out, rows, row_width, width, k, eps, wd, wd_dtype, eps_d);
  else if (dtype == IX_BF16)
    hipLaunchKernelGGL(moe_combine_add_rmsnorm_kernel<bf16_t>, grid, block, smem, stream, (float*)h,
                       (const bf16_t*)y, dest, topk_w, (const bf16_t*)shared, shared_gate, w, w_dtype, (bf16_t*)out,
                       rows, row_width, width, k, eps, wd, wd_dtype, eps_d);
  else
    IX_REQUIRE(false, "dtype must be float32 or bfloat16");
  return ix_check_launch("ix_moe_combine_add_rmsnorm");
}
