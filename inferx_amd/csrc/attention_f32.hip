// Paged attention on the matrix cores in float32, for prompt portions and decoding alike; the same arithmetic as the
// plain kernel (attention_plain.hip): keys [start, p] through the block table, `start` by `span`, scores * scale (then
// capped), softmax online, every product, sum and exponential in 32 bits (v_mfma_f32_16x16x4_f32, expf).
//
// What bounds it: the keys' and values' way from memory in decoding.  The plain kernel has one workgroup per (token,
// head) whose threads each read a key's row from end to end (a cache line per lane and load) and then walk the values
// a key at a time.  Here the unit of work is one wavefront, as in attention_mfma.hip: up to sixteen consecutive queries
// of one request and one query head, or (GQ) the query heads of one token that share a key/value head, over one slice
// of the keys; no LDS, no barrier.  A round is sixteen keys, which lie in one page (page sizes and slices are multiples
// of sixteen), so a round looks up one page, a round ahead of its loads.
//
//   S^T[key][query]  = K[key][:] . Q[query][:]         A = K rows, B = Q rows: 16 bytes a lane, four lanes a row's 64;
//                                                      product j of a piece multiplies its j-th numbers
//   O^T[d][query]   += V^T[d][key] . P^T[key][query]   lane (n, g) has the scores of keys 4 g + i of query n, which is
//                                                      the B operand of product i; V^T (values lie [d][offset] in a
//                                                      page) gives the same four keys of a column as 16 bytes
//
// With several slices each wavefront leaves (max, sum, unnormalised O), merged by a second kernel.
//
// Measured with 16 heads of 128: 8 tokens on contexts of 300 to 1,200 (90 MB) 29 us and 5 for the merge, against 212 of
// the plain kernel; two prompts of 150 and 361 tokens 38 + 6 against 397.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define AF_KEYS 16  // keys per round

// head_dim = 16 NB.  MANY: a tile may hold several queries (tiles of one do without the registers of that case: a decoding
// step of eight requests, 4 layers, takes 1,353 us, with them 1,391)
template <int NB, bool GQ, bool MANY>
__global__ void __launch_bounds__(256)
attn_f32_kernel(const float* q, const float* k_cache, const float* v_cache, const int32_t* __restrict__ block_table,
                const int32_t* __restrict__ tile_seq, const int32_t* __restrict__ tile_q0,
                const int32_t* __restrict__ tile_rows, const int32_t* __restrict__ positions, float* __restrict__ out,
                float* __restrict__ part_o, float* __restrict__ part_ml, int n_tiles, int n_splits, int heads,
                int kv_heads, int page_size, int max_blocks, float scale, int span, const float* __restrict__ sink,
                float softcap) {
  constexpr int D = 16 * NB;
  constexpr bool AHEAD = NB <= 6;  // the next round's keys and values on their way while this one is multiplied
  const int lane = threadIdx.x & 63;
  const int unit = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (unit >= n_tiles * n_splits) return;
  const int tile = unit / n_splits, split = unit - tile * n_splits;
  const int group = heads / kv_heads;
  const int kvh = GQ ? blockIdx.y : blockIdx.y / group;
  const int n = lane & 15, g = lane >> 4;
  const int head = GQ ? kvh * group + min(n, group - 1) : blockIdx.y;
  const int tq0 = tile_q0[tile];
  const int rows = GQ ? group : tile_rows[tile];  // columns of the tile that hold a query
  const int pos0 = positions[tq0];
  const int32_t* table = block_table + static_cast<int64_t>(tile_seq[tile]) * max_blocks;

  // keys that this tile reads at all: [lo, hi); this wavefront's slice [ks, ke)
  const int lo = ix_first_key(pos0, span);
  const int hi = pos0 + (GQ ? 1 : rows);
  const int lo_al = lo & ~(AF_KEYS - 1);
  const int per = ((hi - lo_al + n_splits - 1) / n_splits + AF_KEYS - 1) & ~(AF_KEYS - 1);
  const int ks = lo_al + split * per, ke = min(hi, ks + per);

  const bool my_row = n < rows;
  const int64_t token = tq0 + (GQ || !my_row ? 0 : n);
  f32x4 qf[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c)
    qf[c] = my_row ? *reinterpret_cast<const f32x4*>(q + (token * heads + head) * D + 16 * c + 4 * g)
                   : f32x4{0.f, 0.f, 0.f, 0.f};
  const int my_pos = pos0 + (GQ ? 0 : n);
  const int my_lo = GQ ? lo : ix_first_key(my_pos, span);
  const int last_lo = GQ ? lo : ix_first_key(pos0 + rows - 1, span);  // the first key of the tile's last query

  f32x4 o[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) o[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool sunk = sink != nullptr && split == 0;
  float m = sunk ? sink[head] : -INFINITY;
  float lsum = (sunk && g == 0) ? 1.f : 0.f;  // a column's sum is spread over its four lanes

  auto page_at = [&](int kb) { return max(table[min(kb, hi - 1) / page_size], 0); };  // (a page the window has passed: masked)
  auto load = [&](int kb, int page, f32x4 (&kf)[NB], f32x4 (&vf)[NB]) {
    const int off = kb % page_size;
    const int64_t at = (static_cast<int64_t>(page) * kv_heads + kvh) * page_size * D;
    const float* kr = k_cache + at + (off + n) * D + 4 * g;
    const float* vr = v_cache + at + n * page_size + off + 4 * g;
#pragma unroll
    for (int c = 0; c < NB; ++c) kf[c] = *reinterpret_cast<const f32x4*>(kr + 16 * c);
#pragma unroll
    for (int b = 0; b < NB; ++b) vf[b] = *reinterpret_cast<const f32x4*>(vr + 16 * b * page_size);
  };
  auto round = [&](int kb, const f32x4 (&kf)[NB], f32x4 (&vf)[NB]) {
    f32x4 s0 = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][j], qf[c][j], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][j + 1], qf[c][j + 1], s1, 0, 0, 0);
      }
    float sv[4], mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = kb + 4 * g + i;
      float s = (s0[i] + s1[i]) * scale;
      if (softcap > 0.f) s = softcap * tanhf(s / softcap);
      sv[i] = (my_row && key >= my_lo && key <= my_pos && key < ke) ? s : -INFINITY;
      mx = fmaxf(mx, sv[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;
    if (__any(m_new > m)) {
      const float alpha = expf(m - m_safe);  // (exp(-inf) = 0)
      lsum *= alpha;
#pragma unroll
      for (int b = 0; b < NB; ++b) o[b] *= alpha;
      m = m_new;
    }
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = expf(sv[i] - m_safe);
      lsum += p[i];
    }
    // What lies past the tile's last key, or before its first one, has probability zero, but zero times whatever an
    // earlier request left there need not be zero.
    if (kb + AF_KEYS > hi || kb < lo) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kb + 4 * g + i;
        if (key >= hi || key < lo) {
#pragma unroll
          for (int b = 0; b < NB; ++b) vf[b][i] = 0.f;
        }
      }
    }
    // Likewise a key of the request itself that some queries of the tile see and others do not: where its value is not
    // finite, the others' zero weights would take it up.
    if (MANY && rows > 1 && (kb + AF_KEYS - 1 > pos0 || kb < last_lo)) {
      float z = 0.f;  // (0 or NaN)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) z = fmaf(vf[b][i], 0.f, z);
      if (__any(z != 0.f)) {
        f32x4 seen;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = kb + 4 * g + i;
          seen[i] = key >= my_lo && key <= my_pos ? 1.f : 0.f;
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          f32x4 clean = o[b], count = f32x4{0.f, 0.f, 0.f, 0.f};  // without such values; how many of them a query sees
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const bool odd = !(vf[b][i] * 0.f == 0.f);
            clean = __builtin_amdgcn_mfma_f32_16x16x4f32(odd ? 0.f : vf[b][i], p[i], clean, 0, 0, 0);
            count = __builtin_amdgcn_mfma_f32_16x16x4f32(odd ? 1.f : 0.f, seen[i], count, 0, 0, 0);
            o[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][i], p[i], o[b], 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) o[b][i] = count[i] > 0.f ? o[b][i] : clean[i];
        }
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b) o[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][i], p[i], o[b], 0, 0, 0);
  };

  if (ks < ke) {
    int page = page_at(ks);
    if constexpr (AHEAD) {
      // two register sets that change places; a round past the end is asked for again and not worked
      f32x4 ka[NB], va[NB], kb_[NB], vb[NB];
      load(ks, page, ka, va);
      page = page_at(ks + AF_KEYS);
      for (int kb = ks; kb < ke; kb += 2 * AF_KEYS) {
        const int second = min(kb + AF_KEYS, ke - 1) & ~(AF_KEYS - 1), third = min(kb + 2 * AF_KEYS, ke - 1) & ~(AF_KEYS - 1);
        load(second, kb + AF_KEYS < ke ? page : page_at(second), kb_, vb);
        page = page_at(third);
        __builtin_amdgcn_sched_barrier(0);
        round(kb, ka, va);
        __builtin_amdgcn_sched_barrier(0);
        load(third, page, ka, va);
        page = page_at(third + AF_KEYS);
        __builtin_amdgcn_sched_barrier(0);
        if (kb + AF_KEYS < ke) round(kb + AF_KEYS, kb_, vb);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      for (int kb = ks; kb < ke; kb += AF_KEYS) {
        f32x4 ka[NB], va[NB];
        load(kb, page, ka, va);
        page = page_at(kb + AF_KEYS);
        round(kb, ka, va);
      }
    }
  }

  float l = lsum;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (!my_row) return;
  // lane holds O^T rows d = 16 b + 4 g + i of column n
  if (n_splits == 1) {
    float* dst = out + (token * heads + head) * D + 4 * g;
#pragma unroll
    for (int b = 0; b < NB; ++b)
      *reinterpret_cast<f32x4*>(dst + 16 * b) = f32x4{o[b][0] / l, o[b][1] / l, o[b][2] / l, o[b][3] / l};
  } else {
    const int64_t p = (token * heads + head) * n_splits + split;
    float* dst = part_o + p * D + 4 * g;
#pragma unroll
    for (int b = 0; b < NB; ++b) *reinterpret_cast<f32x4*>(dst + 16 * b) = o[b];
    if (g == 0) {
      part_ml[2 * p] = m;
      part_ml[2 * p + 1] = l;
    }
  }
}

// out[t, h, :] = sum_s o_s e^(m_s - M) / sum_s l_s e^(m_s - M),  M = max_s m_s; a workgroup of 64 per (token, head)
__global__ void __launch_bounds__(64)
attn_f32_combine_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml, float* __restrict__ out,
                        int n_splits, int head_dim) {
  __shared__ float wgt[256];
  const int64_t th = blockIdx.x;
  const float* ml = part_ml + th * n_splits * 2;
  float mloc = -INFINITY;
  for (int s = threadIdx.x; s < n_splits; s += 64) mloc = fmaxf(mloc, ml[2 * s]);
  const float M = ix_wave_max(mloc);
  float lloc = 0.f;
  for (int s = threadIdx.x; s < n_splits; s += 64) {
    const float w = ml[2 * s] == -INFINITY ? 0.f : expf(ml[2 * s] - M);
    wgt[s] = w;
    lloc += w * ml[2 * s + 1];
  }
  const float L = ix_wave_sum(lloc);
  __syncthreads();
  const f32x4* po = reinterpret_cast<const f32x4*>(part_o + th * n_splits * head_dim);
  const int quads = head_dim / 4;
  for (int d = threadIdx.x; d < quads; d += 64) {
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < n_splits; ++s) acc += wgt[s] * po[static_cast<int64_t>(s) * quads + d];
    reinterpret_cast<f32x4*>(out + th * head_dim)[d] = f32x4{acc[0] / L, acc[1] / L, acc[2] / L, acc[3] / L};
  }
}

// Arguments as ix_attention_mfma (float32 throughout; tiles of up to 16 queries; grouped: tiles of one token, the query
// heads of a key/value head together); sink, softcap as in attention_plain.hip.  Workspace when n_splits > 1: part_o
// float32 [tokens * heads * n_splits * head_dim], part_ml float32 [tokens * heads * n_splits * 2].
extern "C" int ix_attention_f32(const float* q, const float* k_cache, const float* v_cache, const int32_t* block_table,
                                const int32_t* tile_seq, const int32_t* tile_q0, const int32_t* tile_rows,
                                const int32_t* positions, float* out, float* part_o, float* part_ml, int64_t tokens,
                                int n_tiles, int n_splits, int heads, int kv_heads, int head_dim, int page_size,
                                int max_blocks, float scale, int span, int grouped, const float* sink, float softcap,
                                hipStream_t stream) {
  IX_REQUIRE(softcap >= 0.f, "the cap of the scores must not be negative");
  IX_REQUIRE(tokens >= 0 && n_tiles >= 0 && heads > 0 && kv_heads > 0 && max_blocks > 0, "sizes must be positive");
  IX_REQUIRE(heads % kv_heads == 0, "heads must be a multiple of kv_heads");
  IX_REQUIRE(head_dim % 16 == 0 && head_dim >= 16 && head_dim <= 256, "head_dim must be a multiple of 16 up to 256");
  IX_REQUIRE(page_size % 16 == 0 && page_size > 0, "page_size must be a multiple of 16");
  IX_REQUIRE(n_splits >= 1 && n_splits <= 256, "n_splits must be between 1 and 256");
  IX_REQUIRE(n_splits == 1 || (part_o != nullptr && part_ml != nullptr), "workspace needed for split keys");
  IX_REQUIRE(heads <= 65535, "too many heads");
  IX_REQUIRE(!grouped || heads / kv_heads <= 16, "grouped queries: at most 16 query heads per key/value head");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache) |
               reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(part_o)) & 15) == 0,
             "operands must lie on 16-byte boundaries");
  if (n_tiles == 0 || tokens == 0) return 0;
  IX_REQUIRE(static_cast<int64_t>(n_tiles) * n_splits < (int64_t(1) << 31) - 4, "too many wavefronts");
  const int units = n_tiles * n_splits, lines = grouped ? kv_heads : heads;
  // four wavefronts per workgroup, fewer while that makes fewer than two workgroups per compute unit
  const int64_t waves = static_cast<int64_t>(units) * lines;
  const int per_group = waves >= 4 * 512 ? 4 : (waves >= 2 * 512 ? 2 : 1);
  dim3 grid((units + per_group - 1) / per_group, lines), block(64 * per_group);
#define CASE(NB)                                                                                                     \
  case NB:                                                                                                           \
    if (grouped)                                                                                                     \
      hipLaunchKernelGGL((attn_f32_kernel<NB, true, false>), grid, block, 0, stream, q, k_cache, v_cache, block_table, tile_seq, \
                         tile_q0, tile_rows, positions, out, part_o, part_ml, n_tiles, n_splits, heads, kv_heads,    \
                         page_size, max_blocks, scale, span, sink, softcap);                                         \
    else if (n_tiles >= tokens) /* tiles of one query each */                                                         \
      hipLaunchKernelGGL((attn_f32_kernel<NB, false, false>), grid, block, 0, stream, q, k_cache, v_cache, block_table, tile_seq, \
                         tile_q0, tile_rows, positions, out, part_o, part_ml, n_tiles, n_splits, heads, kv_heads,    \
                         page_size, max_blocks, scale, span, sink, softcap);                                         \
    else                                                                                                             \
      hipLaunchKernelGGL((attn_f32_kernel<NB, false, true>), grid, block, 0, stream, q, k_cache, v_cache, block_table, tile_seq, \
                         tile_q0, tile_rows, positions, out, part_o, part_ml, n_tiles, n_splits, heads, kv_heads,    \
                         page_size, max_blocks, scale, span, sink, softcap);                                         \
    break;
  switch (head_dim / 16) {
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
    CASE(9) CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) CASE(15) CASE(16)
  }
#undef CASE
  if (ix_check_launch("ix_attention_f32")) return 1;
  if (n_splits > 1) {
    hipLaunchKernelGGL(attn_f32_combine_kernel, dim3(static_cast<unsigned>(tokens * heads)), dim3(64), 0, stream, part_o,
                       part_ml, out, n_splits, head_dim);
    return ix_check_launch("ix_attention_f32");
  }
  return 0;
}
