// Attention over the compressed cache (see latent_attention.hip) for steps whose requests bring their whole contexts, on keys
// and values of every head's own that the caller has formed: bfloat16, keys of 128 + 64 rotated numbers, values of 128.
//
//     kv   [tokens, heads * 256]   the heads' keys, 128 numbers each, then the heads' values
//     rot  [tokens, 64]            the rotated numbers that all heads share
//
// On the latents a pair of a query and a key costs a head 2 (576 + 512) operations, on its own keys and values 2 (192 + 128),
// and to form them costs as much as to move queries and results to the latents and back, which falls away.  Where a context is
// already in the cache (decoding, a later portion) it would all have to be formed anew: there latent_prefill.hip works.
//
// A workgroup takes up to 64 consecutive queries of one request and one head, and its four wavefronts (one a SIMD, 512
// registers each) share out the keys: wavefront w the steps of 32 keys w, w + 4, ..  A wavefront takes every operand that it
// reads from LDS through two products, so LDS gives half of what it could; it loads its own keys and values into two buffers of
// its own (20 KB each, all 160 KB in all), one step ahead, and meets the others only when all have gone through their keys and
// their sums are put together in LDS.
//
//     S^T[key][query] = K Q^T    (v_mfma_f32_32x32x16_bf16; A = key rows, B = queries, in registers throughout)
//     O^T[d][query]  += V^T P^T  (A = value rows, transposed on the way out of LDS, B = the weights)
//
// A lane holds the scores of keys 8 c + 4 h + e of its query (h = lane / 32; c, e < 4): per sixteen keys the eight that it must
// supply to the second product if that takes the keys in this order, which the transposing reads (ds_read_b64_tr_b16, four keys
// at a time) are free to.  The products of the second 32 queries stand beside the exponentials of the first, and the first's
// sums beside the second's exponentials.
//
// 16 heads, one prompt of 2,048 tokens: 46.6 us (460 TFLOP/s; the keys and values of 64 queries come from the die's cache at
// 55 GB/s a compute unit for 24 of them) and 19.2 for the product that forms keys and values, against 154 for latent_prefill.hip
// and 35.5 for the products that move queries and results.
//
// Tiles come in the order of falling work: a workgroup that ends early makes room for the next one.  Pieces of 16 bytes are
// permuted within the rows of LDS so that the sixteen lanes that are served together touch all banks.
#include "common.h"
#include "lds_loads.h"

typedef __bf16 lw_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 lw_bf16x4 __attribute__((ext_vector_type(4)));
typedef float lw_f32x4 __attribute__((ext_vector_type(4)));
typedef float lw_f32x16 __attribute__((ext_vector_type(16)));
typedef short lw_s16x4 __attribute__((ext_vector_type(4)));

#define LW_QUERIES 64
#define LW_KEYS 32                            // keys of a step
#define LW_ROT (LW_KEYS * 256)                // bytes: the rotated numbers behind the keys' own,
#define LW_VALUES (LW_ROT + LW_KEYS * 128)    // the values behind them
#define LW_BUFFER (LW_VALUES + LW_KEYS * 256)
#define LW_LDS (4 * 2 * LW_BUFFER)

__device__ __forceinline__ lw_s16x4 lw_read_turned(const char* at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lw_s16x4*)at);
}

__global__ void __launch_bounds__(256, 1)
latent_whole_kernel(const __bf16* __restrict__ q, int64_t q_t, int64_t q_h, const char* __restrict__ kv,
                    const char* __restrict__ rot, const int32_t* __restrict__ tiles, int n_tiles, __bf16* __restrict__ out,
                    int64_t out_t, int64_t out_h, int heads, float scale_log2) {
  extern __shared__ __attribute__((aligned(1024))) char lw_lds[];
  const int lane = threadIdx.x & 63, qn = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (heads side by side: with a multiple of eight of them all tiles of a head read its keys through one die's cache)
  const int head = static_cast<int>(blockIdx.x) % heads, tile = static_cast<int>(blockIdx.x) / heads;
  const int r0 = tiles[tile], rows = tiles[n_tiles + tile], pos0 = tiles[2 * n_tiles + tile];
  const int hi = pos0 + rows;  // keys that the tile reads
  const unsigned kv_row = static_cast<unsigned>(heads) * 512u;
  const char* const kv_at = kv + static_cast<int64_t>(r0 - pos0) * kv_row + head * 256;
  const char* const rot_at = rot + static_cast<int64_t>(r0 - pos0) * 128;

  // One instruction brings four rows of keys or values or eight of rotated numbers, in the order of the lanes, so it is the
  // lanes' source pieces that are permuted: keys p ^ (row % 16), rotated numbers p ^ (row / 2 % 8), values p ^ 2 (row % 8).
  auto bring = [&](int k0, int buf) {
    const unsigned dst = static_cast<unsigned>(wave * 2 + buf) * LW_BUFFER;
    int ln = lane;  // (hidden once a step: the places would otherwise be worked out before the loop and kept in registers)
    asm volatile("" : "+v"(ln));
    const int r4 = ln >> 4, p4 = ln & 15, r8 = ln >> 3, p8 = ln & 7;
    // keys past the tile's last one are replaced by it: what they would add is masked
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const unsigned row = min(k0 + 4 * i + r4, hi - 1);
      lds_load16<false>(lw_lds, dst + 1024 * i, __umul24(row, kv_row) + ((p4 ^ (4 * (i & 3) + r4)) << 4), kv_at);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned row = min(k0 + 8 * i + r8, hi - 1);
      lds_load16<false>(lw_lds, dst + LW_ROT + 1024 * i, row * 128u + ((p8 ^ (4 * (i & 1) + (r8 >> 1))) << 4), rot_at);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const unsigned row = min(k0 + 4 * i + r4, hi - 1);
      lds_load16<false>(lw_lds, dst + LW_VALUES + 1024 * i, __umul24(row, kv_row) + ((p4 ^ (2 * (4 * (i & 1) + r4))) << 4),
                        kv_at + heads * 256);
    }
  };
  int k0 = LW_KEYS * wave, buf = 0;
  if (k0 < hi) bring(k0, 0);

  lw_bf16x8 qf[2][12];  // B operands: column qn, numbers 16 s + 8 h + j
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const bool on = 32 * b + qn < rows;
    const __bf16* from = q + static_cast<int64_t>(r0 + min(32 * b + qn, rows - 1)) * q_t + head * q_h + 8 * h;
#pragma unroll
    for (int s = 0; s < 12; ++s) {
      qf[b][s] = *reinterpret_cast<const lw_bf16x8*>(from + 16 * s);
      if (!on)
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[b][s][j] = (__bf16)0.f;
    }
  }
  lw_f32x16 zero, o[2][4];
#pragma unroll
  for (int i = 0; i < 16; ++i) zero[i] = 0.f;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[b][d][i] = 0.f;
  float m[2] = {-1e30f, -1e30f}, l[2] = {0.f, 0.f};  // (a query's sum is spread over its two lanes until the end)

  for (; k0 < hi; k0 += 4 * LW_KEYS, buf ^= 1) {
    // Queries, sums and the zero that scores start from live in accumulation registers, from which the products take them;
    // told so at every step, the compiler moves none of them through the others.
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int i = 0; i < 12; ++i) asm volatile("" : "+a"(qf[b][i]));
#pragma unroll
      for (int d = 0; d < 4; ++d) asm volatile("" : "+a"(o[b][d]));
    }
    asm volatile("" : "+a"(zero));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the step before has read its buffer, which the next step's rows take
    if (k0 + 4 * LW_KEYS < hi) {
      bring(k0 + 4 * LW_KEYS, buf ^ 1);
      wait_loads<20>();
    } else {
      wait_loads<0>();
    }
    const char* const at = lw_lds + (wave * 2 + buf) * LW_BUFFER;
    const char* const k_at = at + qn * 256;
    const char* const t_at = at + LW_ROT + qn * 128;
    lw_bf16x8 ka[12];
#pragma unroll
    for (int s = 0; s < 8; ++s) ka[s] = *reinterpret_cast<const lw_bf16x8*>(k_at + (((2 * s + h) ^ (qn & 15)) << 4));
#pragma unroll
    for (int s = 0; s < 4; ++s) ka[8 + s] = *reinterpret_cast<const lw_bf16x8*>(t_at + (((2 * s + h) ^ ((qn >> 1) & 7)) << 4));
    lw_f32x16 s[2];
#pragma unroll
    for (int i = 0; i < 12; ++i) s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[i], qf[0][i], i ? s[0] : zero, 0, 0, 0);

    // The reference point m of the exponentials (in units of log2) follows the running maximum lazily: it moves only when the
    // maximum has outgrown it by more than 2^8.  Any m gives the same quotient.
    auto mask_and_refer = [&](int b) {
      if (k0 + LW_KEYS - 1 > pos0 + 32 * b) {  // (the diagonal)
        const int last = pos0 + 32 * b + qn - k0 - 4 * h;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] = 8 * (i >> 2) + (i & 3) <= last ? s[b][i] : -INFINITY;
      }
      float mx = fmaxf(s[b][0], s[b][1]);
#pragma unroll
      for (int i = 2; i < 16; i += 2) mx = fmaxf(mx, fmaxf(s[b][i], s[b][i + 1]));
      if (__any(mx * scale_log2 > m[b] + 8.f)) {
        const float top = fmaxf(mx, __shfl_xor(mx, 32)) * scale_log2, m_new = fmaxf(m[b], top);
        const float alpha = __builtin_amdgcn_exp2f(m[b] - m_new);
        l[b] *= alpha;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          lw_f32x16 v = o[b][d];
          asm volatile("" : "+v"(v));
#pragma unroll
          for (int i = 0; i < 16; ++i) v[i] *= alpha;
          asm volatile("" : "+a"(v));
          o[b][d] = v;
        }
        m[b] = m_new;
      }
    };
    lw_bf16x8 pf[2][2];
    auto weigh = [&](int b) {
      float sum[2] = {0.f, 0.f};
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[b][8 * g + j], scale_log2, -m[b]));
          sum[j & 1] += p;
          pf[b][g][j] = (__bf16)p;
        }
      l[b] += sum[0] + sum[1];
      asm volatile("" : "+v"(pf[b][0]), "+v"(pf[b][1]), "+v"(l[b]));  // (here, not where they are used)
    };
    mask_and_refer(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 12; ++i) s[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[i], qf[1][i], i ? s[1] : zero, 0, 0, 0);
    weigh(0);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one product, then some of the exponentials' work
      __builtin_amdgcn_sched_group_barrier(0x402, 6, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // values: lane group of sixteen G takes d 16 (G % 2) .. of a block of 32 and keys 4 h + e (then 8 + 4 h + e) of sixteen
    lw_bf16x8 va[2][4];
    {
      const int e = (lane >> 2) & 3, x = 2 * (4 * h + e), in = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
      const char* const v_at = at + LW_VALUES + (4 * h + e) * 256 + 8 * (lane & 1);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const char* from = v_at + (((4 * d + in) ^ x) << 4);
#pragma unroll
        for (int g = 0; g < 2; ++g)
          va[g][d] = __builtin_bit_cast(lw_bf16x8, __builtin_shufflevector(lw_read_turned(from + 16 * g * 256),
                                                                           lw_read_turned(from + (16 * g + 8) * 256), 0, 1, 2, 3,
                                                                           4, 5, 6, 7));
      }
    }
    mask_and_refer(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int d = 0; d < 4; ++d) o[0][d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[g][d], pf[0][g], o[0][d], 0, 0, 0);
    weigh(1);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x402, 9, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int d = 0; d < 4; ++d) o[1][d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[g][d], pf[1][g], o[1][d], 0, 0, 0);
  }

  // The wavefronts' sums, each in its own buffers: [query block][block of 32 numbers][c][lane] of four numbers, then the
  // reference points and sums of the weights; wavefront w puts numbers 32 w .. together.
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  {
    char* const mine = lw_lds + wave * 2 * LW_BUFFER;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          *reinterpret_cast<lw_f32x4*>(mine + (((b * 4 + d) * 4 + c) * 64 + lane) * 16) =
              lw_f32x4{o[b][d][4 * c], o[b][d][4 * c + 1], o[b][d][4 * c + 2], o[b][d][4 * c + 3]};
      const float sum = l[b] + __shfl_xor(l[b], 32);
      *reinterpret_cast<float2*>(mine + 32768 + (b * 64 + lane) * 8) = make_float2(m[b], sum);
    }
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float2 ml[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) ml[w] = *reinterpret_cast<const float2*>(lw_lds + w * 2 * LW_BUFFER + 32768 + (b * 64 + lane) * 8);
    const float top = fmaxf(fmaxf(ml[0].x, ml[1].x), fmaxf(ml[2].x, ml[3].x));
    float by[4], sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      by[w] = __builtin_amdgcn_exp2f(ml[w].x - top);
      sum += by[w] * ml[w].y;
    }
    const float inv = 1.0f / sum;
    if (32 * b + qn >= rows) continue;
    __bf16* const to = out + static_cast<int64_t>(r0 + 32 * b + qn) * out_t + head * out_h + 32 * wave + 4 * h;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      lw_f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const lw_f32x4 part = *reinterpret_cast<const lw_f32x4*>(lw_lds + w * 2 * LW_BUFFER + (((b * 4 + wave) * 4 + c) * 64 + lane) * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = fmaf(part[e], by[w], v[e]);
      }
      lw_bf16x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = static_cast<__bf16>(v[e] * inv);
      *reinterpret_cast<lw_bf16x4*>(to + 8 * c) = r;
    }
  }
}

// tiles int32 [3, n_tiles]: a tile's first row, its rows (1 .. 64) and the position of the first; a request's rows are its
// positions 0, 1, .. one after the other.  q (and out) element (t, h, i) at q[t * q_t + h * q_h + i], rows on 16-byte (8-byte)
// boundaries.
extern "C" int ix_latent_whole(const void* q, int64_t q_t, int64_t q_h, const void* kv, const void* rot, const int32_t* tiles,
                               int n_tiles, void* out, int64_t out_t, int64_t out_h, int64_t tokens, int heads, float scale,
                               hipStream_t stream) {
  IX_REQUIRE(n_tiles >= 0 && heads > 0 && tokens >= 0, "sizes must be positive");
  // (a row's number and its bytes are multiplied as numbers of 24 bits)
  IX_REQUIRE(tokens < (1 << 24) && heads < (1 << 15), "up to 2^24 tokens and 2^15 heads, less one each");
  IX_REQUIRE(tokens * heads * 512 < (int64_t(1) << 32), "places within keys and values must fit 32 bits");
  IX_REQUIRE((q_t | q_h) % 8 == 0 && (out_t | out_h) % 4 == 0, "rows of queries on 16-byte, of results on 8-byte boundaries");
  IX_REQUIRE(static_cast<int64_t>(n_tiles) * heads < (int64_t(1) << 31), "too many workgroups for one launch");
  if (n_tiles == 0) return 0;
  static bool raised = false;
  if (!raised) {
    // (a refusal shows as the launch's own error)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(latent_whole_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, LW_LDS);
    (void)hipGetLastError();
    raised = true;
  }
  hipLaunchKernelGGL(latent_whole_kernel, dim3(static_cast<unsigned>(n_tiles) * heads), dim3(256), LW_LDS, stream, (const __bf16*)q,
                     q_t, q_h, (const char*)kv, (const char*)rot, tiles, n_tiles, (__bf16*)out, out_t, out_h, heads,
                     scale * 1.4426950408889634f);
  return ix_check_launch("ix_latent_whole");
}
