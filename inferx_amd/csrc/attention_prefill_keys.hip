// Paged attention for prompt portions (bfloat16, heads of 128), a tile's keys shared out among the wavefronts.
//
// attention_prefill128.hip gives a wavefront 32 queries of a tile of 128 and all keys.  A prompt of some thousand tokens then has
// fewer tiles than the chip has compute units to give them to, or just as many, and all wait for the tile that reads most keys
// (2,048 tokens of 16 heads: 256 workgroups, of which the longest has twice the average).  Here a workgroup takes 64 queries of
// one request and one head, so there are twice as many tiles with half the work, and its four wavefronts (one a SIMD, 512 registers
// each) take the steps of 32 keys w, w + 4, .. of them: the structure of latent_whole.hip, where it is explained, on the pages of
// the cache.  Keys and values are loaded for 64 queries instead of 128, which is what bounds it where there are tiles enough.
// Tiles of 128 / this, us: 16 heads, a prompt of 130 tokens 11.9 / 9.7, of 1,024 32.5 (in two slices) / 20.0, of 2,048 48.4 / 39.3 (in a
// step, where weights have passed through the caches since, 54.4 / 46.6), of 4,096 98.9 / 113.6 (there the caller stays with tiles of 128).  Error against 64 bits, of the norm, same sizes: 1.90e-3 / 1.87e-3,
// 2,048 tokens 2.09e-3 / 2.04e-3.
#include "common.h"
#include "lds_loads.h"

typedef __bf16 pk_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 pk_bf16x4 __attribute__((ext_vector_type(4)));
typedef float pk_f32x4 __attribute__((ext_vector_type(4)));
typedef float pk_f32x16 __attribute__((ext_vector_type(16)));

#define PK_QUERIES 64
#define PK_KEYS 32                     // keys of a step
#define PK_VALUES (PK_KEYS * 256)      // bytes: the values behind the keys
#define PK_BUFFER (2 * PK_VALUES)
#define PK_PART (32768 + 1024)         // bytes that a wavefront's sums take at the end
#define PK_LDS (4 * PK_PART)

__global__ void __launch_bounds__(256, 1)
attn_prefill_keys_kernel(const __bf16* __restrict__ q, const char* __restrict__ k_cache, const char* __restrict__ v_cache,
                         const int32_t* __restrict__ block_table, const int32_t* __restrict__ tiles, int n_tiles,
                         const int32_t* __restrict__ positions, __bf16* __restrict__ out, int heads, int kv_heads,
                         int page_shift, int max_blocks, float scale_log2) {
  extern __shared__ __attribute__((aligned(1024))) char pk_lds[];
  const int lane = threadIdx.x & 63, qn = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (heads side by side: with a multiple of eight of them all tiles of a head read its keys through one die's cache)
  const int head = static_cast<int>(blockIdx.x) % heads, tile = static_cast<int>(blockIdx.x) / heads;
  const int r0 = tiles[n_tiles + tile], rows = tiles[2 * n_tiles + tile], pos0 = positions[r0];
  const int hi = pos0 + rows;  // keys that the tile reads
  const int32_t* const table = block_table + static_cast<int64_t>(tiles[tile]) * max_blocks;
  const int kvh = head / (heads / kv_heads), last_page = (hi - 1) >> page_shift, in_page = (1 << page_shift) - 1;

  // A step's two groups of sixteen keys lie in a page each.  One instruction brings four rows of keys, or 32 rows of transposed
  // values with sixteen keys each, in the order of the lanes, so it is the lanes' source pieces that are permuted: keys
  // p ^ (row % 16), values p ^ (d / 8 % 2).  Pages are named a step before they are asked for; a group past the last key takes
  // the last page instead.
  int page[2];
  auto name_pages = [&](int k0) {
#pragma unroll
    for (int g = 0; g < 2; ++g) page[g] = table[min((k0 + 16 * g) >> page_shift, last_page)];
  };
  auto bring = [&](int k0, int buf) {
    const unsigned dst = static_cast<unsigned>(wave * 2 + buf) * PK_BUFFER;
    int ln = lane;  // (hidden once a step: the places would otherwise be worked out before the loop and kept in registers)
    asm volatile("" : "+v"(ln));
    const unsigned r4 = ln >> 4, p4 = ln & 15, d32 = ln >> 1, p2 = ln & 1;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int off = (k0 + 16 * g) & in_page;
      const char* const from = k_cache + (((static_cast<int64_t>(page[g]) * kv_heads + kvh) << page_shift) + off) * 256;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        lds_load16<false>(pk_lds, dst + 4096 * g + 1024 * i, (4 * i + r4) * 256 + ((p4 ^ (4 * i + r4)) << 4), from);
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int off = (k0 + 16 * g) & in_page;
      const char* const from = v_cache + (((static_cast<int64_t>(page[g]) * kv_heads + kvh) * 128) << (page_shift + 1)) + off * 2;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        lds_load16<false>(pk_lds, dst + PK_VALUES + 4096 * g + 1024 * i,
                          ((32 * i + d32) << (page_shift + 1)) + ((p2 ^ ((d32 >> 3) & 1)) << 4), from);
    }
  };
  int k0 = PK_KEYS * wave, buf = 0;
  if (k0 < hi) {
    name_pages(k0);
    bring(k0, 0);
    name_pages(k0 + 4 * PK_KEYS);
  }

  pk_bf16x8 qf[2][8];  // B operands: column qn, numbers 16 s + 8 h + j
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const bool on = 32 * b + qn < rows;
    const __bf16* from = q + (static_cast<int64_t>(r0 + min(32 * b + qn, rows - 1)) * heads + head) * 128 + 8 * h;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      qf[b][s] = *reinterpret_cast<const pk_bf16x8*>(from + 16 * s);
      if (!on)
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[b][s][j] = (__bf16)0.f;
    }
  }
  pk_f32x16 zero, o[2][4];
#pragma unroll
  for (int i = 0; i < 16; ++i) zero[i] = 0.f;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[b][d][i] = 0.f;
  float m[2] = {-1e30f, -1e30f}, l[2] = {0.f, 0.f};  // (a query's sum is spread over its two lanes until the end)

  for (; k0 < hi; k0 += 4 * PK_KEYS, buf ^= 1) {
    // Queries, sums and the zero that scores start from live in accumulation registers, from which the products take them;
    // told so at every step, the compiler moves none of them through the others.
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int i = 0; i < 8; ++i) asm volatile("" : "+a"(qf[b][i]));
#pragma unroll
      for (int d = 0; d < 4; ++d) asm volatile("" : "+a"(o[b][d]));
    }
    asm volatile("" : "+a"(zero));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the step before has read its buffer, which the next step's rows take
    if (k0 + 4 * PK_KEYS < hi) {
      bring(k0 + 4 * PK_KEYS, buf ^ 1);
      name_pages(k0 + 8 * PK_KEYS);
      wait_loads<16>();
    } else {
      wait_loads<0>();
    }
    const char* const at = pk_lds + (wave * 2 + buf) * PK_BUFFER;
    const char* const k_at = at + qn * 256;
    pk_bf16x8 ka[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) ka[s] = *reinterpret_cast<const pk_bf16x8*>(k_at + (((2 * s + h) ^ (qn & 15)) << 4));
    pk_f32x16 s[2];
#pragma unroll
    for (int i = 0; i < 8; ++i) s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[i], qf[0][i], i ? s[0] : zero, 0, 0, 0);

    // The reference point m of the exponentials (in units of log2) follows the running maximum lazily: it moves only when the
    // maximum has outgrown it by more than 2^8.  Any m gives the same quotient.
    auto mask_and_refer = [&](int b) {
      if (k0 + PK_KEYS - 1 > pos0 + 32 * b) {  // (the diagonal)
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
          pk_f32x16 v = o[b][d];
          asm volatile("" : "+v"(v));
#pragma unroll
          for (int i = 0; i < 16; ++i) v[i] *= alpha;
          asm volatile("" : "+a"(v));
          o[b][d] = v;
        }
        m[b] = m_new;
      }
    };
    pk_bf16x8 pf[2][2];
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
    for (int i = 0; i < 8; ++i) s[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[i], qf[1][i], i ? s[1] : zero, 0, 0, 0);
    weigh(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one product, then some of the exponentials' work
      __builtin_amdgcn_sched_group_barrier(0x402, 6, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // values: row 32 d + qn, its keys 4 h + e and 8 + 4 h + e of sixteen
    pk_bf16x8 va[2][4];
    {
      const char* const v_at = at + PK_VALUES + qn * 32 + 8 * h;
      const int first = 16 * ((qn >> 3) & 1);
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const char* from = v_at + 4096 * g + 1024 * d;
          va[g][d] = __builtin_shufflevector(*reinterpret_cast<const pk_bf16x4*>(from + first),
                                             *reinterpret_cast<const pk_bf16x4*>(from + (16 - first)), 0, 1, 2, 3, 4, 5, 6, 7);
        }
      if (k0 + PK_KEYS > hi) {  // whatever lies behind the last key: a weight of zero times that need not be zero
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const bool there = k0 + 16 * g + 8 * (j >> 2) + 4 * h + (j & 3) < hi;
#pragma unroll
            for (int d = 0; d < 4; ++d) va[g][d][j] = there ? va[g][d][j] : (__bf16)0.f;
          }
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

  // The wavefronts' sums, each in a part of LDS: [query block][block of 32 numbers][c][lane] of four numbers, then the
  // reference points and sums of the weights; wavefront w puts numbers 32 w .. together.
  __syncthreads();  // (they reach into each other's)
  {
    char* const mine = pk_lds + wave * PK_PART;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          *reinterpret_cast<pk_f32x4*>(mine + (((b * 4 + d) * 4 + c) * 64 + lane) * 16) =
              pk_f32x4{o[b][d][4 * c], o[b][d][4 * c + 1], o[b][d][4 * c + 2], o[b][d][4 * c + 3]};
      const float sum = l[b] + __shfl_xor(l[b], 32);
      *reinterpret_cast<float2*>(mine + 32768 + (b * 64 + lane) * 8) = make_float2(m[b], sum);
    }
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float2 ml[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) ml[w] = *reinterpret_cast<const float2*>(pk_lds + w * PK_PART + 32768 + (b * 64 + lane) * 8);
    const float top = fmaxf(fmaxf(ml[0].x, ml[1].x), fmaxf(ml[2].x, ml[3].x));
    float by[4], sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      by[w] = __builtin_amdgcn_exp2f(ml[w].x - top);
      sum += by[w] * ml[w].y;
    }
    const float inv = 1.0f / sum;
    if (32 * b + qn >= rows) continue;
    __bf16* const to = out + (static_cast<int64_t>(r0 + 32 * b + qn) * heads + head) * 128 + 32 * wave + 4 * h;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      pk_f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const pk_f32x4 part = *reinterpret_cast<const pk_f32x4*>(pk_lds + w * PK_PART + (((b * 4 + wave) * 4 + c) * 64 + lane) * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = fmaf(part[e], by[w], v[e]);
      }
      pk_bf16x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = static_cast<__bf16>(v[e] * inv);
      *reinterpret_cast<pk_bf16x4*>(to + 8 * c) = r;
    }
  }
}

// tiles int32 [3, n_tiles]: a tile's request, first row and rows (1 .. 64), consecutive positions of the request; pages of a power of
// two of keys from 16 on.  k_cache [pages, kv_heads, page, 128], v_cache [pages, kv_heads, 128, page].
extern "C" int ix_attention_prefill_keys(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_table,
                                         const int32_t* tiles, int n_tiles, const int32_t* positions, void* out, int heads,
                                         int kv_heads, int page_size, int max_blocks, float scale, hipStream_t stream) {
  IX_REQUIRE(n_tiles >= 0 && heads > 0 && kv_heads > 0 && max_blocks > 0, "sizes must be positive");
  IX_REQUIRE(heads % kv_heads == 0, "heads must be a multiple of kv_heads");
  IX_REQUIRE(page_size >= 16 && page_size <= (1 << 20) && (page_size & (page_size - 1)) == 0,
             "page_size must be a power of two from 16 on");
  IX_REQUIRE(static_cast<int64_t>(n_tiles) * heads < (int64_t(1) << 31), "too many workgroups for one launch");
  if (n_tiles == 0) return 0;
  int page_shift = 4;
  while ((1 << page_shift) < page_size) ++page_shift;
  static bool raised = false;
  if (!raised) {
    // (a refusal shows as the launch's own error)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(attn_prefill_keys_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, PK_LDS);
    (void)hipGetLastError();
    raised = true;
  }
  hipLaunchKernelGGL(attn_prefill_keys_kernel, dim3(static_cast<unsigned>(n_tiles) * heads), dim3(256), PK_LDS, stream, (const __bf16*)q,
                     (const char*)k_cache, (const char*)v_cache, block_table, tiles, n_tiles, positions, (__bf16*)out, heads, kv_heads,
                     page_shift, max_blocks, scale * 1.4426950408889634f);
  return ix_check_launch("ix_attention_prefill_keys");
}
