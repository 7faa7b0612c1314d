// Differential attention (attention_diff.hip has the arithmetic) for the prompt portions of a step, on the matrix cores:
// bfloat16, heads and values of 64 or 128.
//
// A workgroup of four wavefronts takes up to 64 consecutive queries of a request, sixteen a wavefront, of one head and
// BOTH its score maps.  Rounds of 32 keys of both maps and their values go through two LDS buffers, one barrier a round,
// the next round's on its way from memory in registers and its pages looked up a round before that.  The operand layouts
// are those of attention_mfma.hip (S^T = K Q^T, O^T += V^T P^T, nothing shuffled).  A wavefront ends up with both maps'
// sums of its queries, so their difference and its norm are formed from registers.
//
// What bounds it: a round's chain of waits (operands out of LDS, products, exponentials, products, barrier: 1.3 us) and, with
// two workgroups on a compute unit, the softmax's vector instructions.  Both maps' products and softmaxes are therefore
// one chain, and the values are read before it.  Against a wavefront per (16 queries, head, map) that reads keys and values
// from L2 for itself and leaves 1 KB a (token, head, map) for a second launch (attention_diff_mfma.hip), us, 16 heads of 64
// on 4 sets of keys, values of 128, a window of 1,024: prompts of 611 and 1,437 48 (91 + 14), 2,048 48 (138), eight of 200 16 (37).
//
// The keys that a tile reads are two runs, rounds number both through: the kept first tokens that lie before the window of
// the tile's first query, and the window's keys up to its last query.
#include "common.h"

typedef __bf16 dp_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 dp_bf16x4 __attribute__((ext_vector_type(4)));
typedef float dp_f32x4 __attribute__((ext_vector_type(4)));

#define DP_KEYS 32     // keys of a round
#define DP_QUERIES 64  // queries of a workgroup

// NB, NBV: sixteens of a key's and a value's numbers (4 or 8)
template <int NB, int NBV>
__global__ void __launch_bounds__(256, 2)
attn_diff_prefill_kernel(const __bf16* __restrict__ q, const __bf16* __restrict__ k_cache, const __bf16* __restrict__ v_cache,
                         const int32_t* __restrict__ block_table, const int32_t* __restrict__ tile_seq,
                         const int32_t* __restrict__ tile_q0, const int32_t* __restrict__ tile_rows,
                         const int32_t* __restrict__ positions, __bf16* __restrict__ out, int n_tiles, int heads,
                         int kv_heads, int page_size, int max_blocks, float scale_log2, int window, int keep_first,
                         int page_shift, float lambda, float eps, float mult) {
  constexpr int D = 16 * NB, V = 16 * NBV, NC = NB / 2;
  constexpr int KP = 2 * NB;                   // 16-byte pieces of a key
  constexpr int NK = DP_KEYS * KP / 256, NV = V * 4 / 256;  // pieces a thread brings of each map's keys, of the values
  constexpr int KTILE = DP_KEYS * D, BUFFER = 2 * KTILE + V * DP_KEYS;
  __shared__ __attribute__((aligned(16))) __bf16 lds[2 * BUFFER];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  // (a tile's heads side by side; the last tiles, which read the most keys of a request, first)
  const int head = static_cast<int>(blockIdx.x) % heads, tile = n_tiles - 1 - static_cast<int>(blockIdx.x) / heads;
  const int kvh = head / (heads / kv_heads);
  const int tq0 = tile_q0[tile], rows = tile_rows[tile], pos0 = positions[tq0];
  const int32_t* table = block_table + static_cast<int64_t>(tile_seq[tile]) * max_blocks;

  const int lo = (window > 0 && pos0 + 1 > window) ? pos0 + 1 - window : 0;
  const int hi = pos0 + rows;
  const int lo_al = lo & ~(DP_KEYS - 1);
  const int kept = min(keep_first, lo);
  const int rounds_kept = min((kept + DP_KEYS - 1) & ~(DP_KEYS - 1), lo_al) / DP_KEYS;
  const int n_rounds = rounds_kept + (hi - lo_al + DP_KEYS - 1) / DP_KEYS;
  auto first_key = [&](int r) {
    r = min(r, n_rounds - 1);  // (past the end: the last round once more, not used)
    return r < rounds_kept ? r * DP_KEYS : lo_al + (r - rounds_kept) * DP_KEYS;
  };

  // this wavefront's queries: w0 .. w0 + w_rows of the tile
  const int w0 = 16 * wave, w_rows = max(0, min(16, rows - w0)), w_pos = pos0 + w0;
  dp_bf16x8 qf[2][NC];
#pragma unroll
  for (int mp = 0; mp < 2; ++mp)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[mp][c][j] = (__bf16)0.f;
      if (n < w_rows)
        qf[mp][c] = *reinterpret_cast<const dp_bf16x8*>(
            q + ((static_cast<int64_t>(tq0 + w0 + n) * heads + head) * 2 + mp) * D + 32 * c + 8 * g);
    }
  dp_f32x4 o[2][NBV];
  float m[2] = {-INFINITY, -INFINITY}, lsum[2] = {0.f, 0.f};
#pragma unroll
  for (int mp = 0; mp < 2; ++mp)
#pragma unroll
    for (int b = 0; b < NBV; ++b) o[mp][b] = dp_f32x4{0.f, 0.f, 0.f, 0.f};

  auto page_of = [&](int key) { return page_shift >= 0 ? key >> page_shift : key / page_size; };
  // Where the pieces of a row lie: sixteen rows that are read at one piece (keys 8 a + b or 8 a + 4 + b, a, b < 4; sixteen
  // consecutive columns of V) fall on different groups of four banks.
  auto k_at = [&](int r, int p) {
    const int swap = KP == 8 ? (((r >> 1) & 1) | (((r >> 3) & 3) << 1)) : ((r & 3) | (((r >> 3) & 3) << 2));
    return r * D + 8 * (p ^ swap);
  };
  auto v_at = [&](int d, int p) { return 2 * KTILE + d * DP_KEYS + 8 * (p ^ ((d >> 2) & 3)); };
  struct Pages { int at[2]; };  // of a round's two sixteens of keys
  struct Set { dp_bf16x8 k[2][NK], v[NV]; };
  auto look_up = [&](int r) {
    const int kb = first_key(r);
    Pages pg;
#pragma unroll
    for (int b = 0; b < 2; ++b) pg.at[b] = max(table[page_of(min(kb + 16 * b, hi - 1))], 0);  // (given back: masked)
    return pg;
  };
  const int64_t k_page = static_cast<int64_t>(2 * kv_heads) * page_size * D, v_page = static_cast<int64_t>(kv_heads) * V * page_size;
  const __bf16* const k_head = k_cache + static_cast<int64_t>(2 * kvh) * page_size * D;
  const __bf16* const v_head = v_cache + static_cast<int64_t>(kvh) * V * page_size;
  auto fetch = [&](int r, const Pages& pg, Set& s) {
    const int kb = first_key(r);
    int off[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int key = min(kb + 16 * b, hi - 1) & ~15;  // (a sixteen past the end: an earlier one once more, masked)
      off[b] = key - page_of(key) * page_size;
    }
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int id = 256 * i + tid, row = id / KP, p = id % KP, b = row >> 4;
      const __bf16* from = k_head + (b ? pg.at[1] : pg.at[0]) * k_page + ((b ? off[1] : off[0]) + (row & 15)) * D + 8 * p;
      s.k[0][i] = *reinterpret_cast<const dp_bf16x8*>(from);
      s.k[1][i] = *reinterpret_cast<const dp_bf16x8*>(from + static_cast<int64_t>(page_size) * D);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int id = 256 * i + tid, d = id >> 2, p = id & 3, b = p >> 1;
      s.v[i] = *reinterpret_cast<const dp_bf16x8*>(v_head + (b ? pg.at[1] : pg.at[0]) * v_page + d * page_size +
                                                   (b ? off[1] : off[0]) + 8 * (p & 1));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto put = [&](const Set& s, __bf16* buf) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int id = 256 * i + tid;
#pragma unroll
      for (int mp = 0; mp < 2; ++mp)
        *reinterpret_cast<dp_bf16x8*>(buf + mp * KTILE + k_at(id / KP, id % KP)) = s.k[mp][i];
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int id = 256 * i + tid;
      *reinterpret_cast<dp_bf16x8*>(buf + v_at(id >> 2, id & 3)) = s.v[i];
    }
  };
  const int w_lo = (window > 0 && w_pos + 1 > window) ? w_pos + 1 - window : 0;
  const int my_pos = w_pos + n;
  const int my_lo = (window > 0 && my_pos + 1 > window) ? my_pos + 1 - window : 0;
  auto multiply = [&](int r, const __bf16* buf) {
    const int kb = first_key(r);
    // (uniform over the wavefront) no query of these sixteen sees the round
    if (w_rows == 0 || kb > w_pos + w_rows - 1 || (kb >= keep_first && window > 0 && kb + DP_KEYS + window <= w_pos + 1)) return;
    const bool inner = w_rows == 16 && kb + DP_KEYS - 1 <= w_pos &&
                       (window == 0 || kb > w_pos + 15 - window || kb + DP_KEYS <= keep_first);
    // (both maps' products first, then both softmaxes: one chain of waits instead of two)
    dp_f32x4 s[2][2];
#pragma unroll
    for (int mp = 0; mp < 2; ++mp) {
      dp_bf16x8 kf[2][NC];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int c = 0; c < NC; ++c)
          kf[b][c] = *reinterpret_cast<const dp_bf16x8*>(buf + mp * KTILE + k_at(8 * (n >> 2) + 4 * b + (n & 3), 4 * c + g));
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        s[mp][b] = dp_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NC; ++c) s[mp][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[b][c], qf[mp][c], s[mp][b], 0, 0, 0);
      }
    }
    dp_bf16x8 vf[NBV];  // (on their way while the weights are worked out)
#pragma unroll
    for (int b = 0; b < NBV; ++b) vf[b] = *reinterpret_cast<const dp_bf16x8*>(buf + v_at(16 * b + n, g));
    __builtin_amdgcn_sched_barrier(0);
    // values of keys that none of these queries may read: zero (their weight is zero, but zero times whatever lies there, or
    // whatever another query may see, need not be)
    if (kb + DP_KEYS > w_pos + w_rows || (kb < w_lo && kb + DP_KEYS > keep_first)) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = kb + 8 * g + j;
        if (key >= w_pos + w_rows || (key < w_lo && key >= keep_first)) {
#pragma unroll
          for (int b = 0; b < NBV; ++b) vf[b][j] = (__bf16)0.f;
        }
      }
    }
    if (!inner) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = kb + 8 * g + j;
        const bool ok = n < w_rows && key <= my_pos && (key >= my_lo || key < keep_first);
#pragma unroll
        for (int mp = 0; mp < 2; ++mp) s[mp][j >> 2][j & 3] = ok ? s[mp][j >> 2][j & 3] : -INFINITY;
      }
    }
    float mx[2];
#pragma unroll
    for (int mp = 0; mp < 2; ++mp) {
      mx[mp] = -INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) mx[mp] = fmaxf(mx[mp], s[mp][j >> 2][j & 3]);
    }
    // The reference point of the exponentials (in units of log2, the same in a column's four lanes) follows the running
    // maximum lazily; whether any column's has outgrown it needs no exchange between the lanes.
    if (__any(mx[0] * scale_log2 > m[0] + 8.f || mx[1] * scale_log2 > m[1] + 8.f)) {
#pragma unroll
      for (int mp = 0; mp < 2; ++mp) {
        float top = mx[mp];
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64)) * scale_log2;
        const float m_new = fmaxf(m[mp], top);
        const float alpha = __builtin_amdgcn_exp2f(m[mp] - ((m_new == -INFINITY) ? 0.f : m_new));
        lsum[mp] *= alpha;
#pragma unroll
        for (int b = 0; b < NBV; ++b) o[mp][b] *= alpha;
        m[mp] = m_new;
      }
    }
    dp_bf16x8 pf[2];
#pragma unroll
    for (int mp = 0; mp < 2; ++mp) {
      const float m_safe = (m[mp] == -INFINITY) ? 0.f : m[mp];
      float psum = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[mp][j >> 2][j & 3], scale_log2, -m_safe));
        psum += p;
        pf[mp][j] = (__bf16)p;
      }
      lsum[mp] += psum;
    }
#pragma unroll
    for (int b = 0; b < NBV; ++b)
#pragma unroll
      for (int mp = 0; mp < 2; ++mp) o[mp][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[b], pf[mp], o[mp][b], 0, 0, 0);
  };

  // round r lies in buffer r & 1; while it is worked, round r + 1 arrives in one register set and r + 2 is asked for
  Set one, two;
  Pages pg = look_up(0);
  fetch(0, pg, one);
  pg = look_up(1);
  fetch(1, pg, two);
  pg = look_up(2);
  put(one, lds);
  __syncthreads();
  for (int r = 0; r < n_rounds; r += 2) {
    fetch(r + 2, pg, one);
    pg = look_up(r + 3);
    multiply(r, lds);
    put(two, lds + BUFFER);
    __syncthreads();
    fetch(r + 3, pg, two);
    pg = look_up(r + 4);
    if (r + 1 < n_rounds) multiply(r + 1, lds + BUFFER);
    put(one, lds);
    __syncthreads();
  }

  float inv[2];
#pragma unroll
  for (int mp = 0; mp < 2; ++mp) {
    float l = lsum[mp];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    inv[mp] = 1.0f / l;
  }
  // lane holds O^T rows 16 b + 4 g + i of column n
  float ss = 0.f;
#pragma unroll
  for (int b = 0; b < NBV; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[0][b][i] = o[0][b][i] * inv[0] - lambda * (o[1][b][i] * inv[1]);
      ss += o[0][b][i] * o[0][b][i];
    }
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (n >= w_rows) return;
  const float f = mult / sqrtf(ss / static_cast<float>(V) + eps);
  __bf16* dst = out + (static_cast<int64_t>(tq0 + w0 + n) * heads + head) * V + 4 * g;
#pragma unroll
  for (int b = 0; b < NBV; ++b)
    *reinterpret_cast<dp_bf16x4*>(dst + 16 * b) =
        dp_bf16x4{(__bf16)(o[0][b][0] * f), (__bf16)(o[0][b][1] * f), (__bf16)(o[0][b][2] * f), (__bf16)(o[0][b][3] * f)};
}

extern "C" int ix_attention_diff_prefill_fits(int head_dim, int value_dim, int page_size) {
  return (head_dim == 64 || head_dim == 128) && (value_dim == 64 || value_dim == 128) && page_size > 0 && page_size % 16 == 0;
}

// Arguments as ix_attention_diff_mfma, tiles of up to 64 queries; no workspace.
extern "C" int ix_attention_diff_prefill(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_table,
                                         const int32_t* tile_seq, const int32_t* tile_q0, const int32_t* tile_rows,
                                         const int32_t* positions, void* out, int64_t tokens, int n_tiles, int heads,
                                         int kv_heads, int head_dim, int value_dim, int page_size, int max_blocks,
                                         float scale, int window, int keep_first, float lambda, float eps, float mult,
                                         hipStream_t stream) {
  IX_REQUIRE(tokens >= 0 && n_tiles >= 0 && heads > 0 && kv_heads > 0 && max_blocks > 0, "sizes must be positive");
  IX_REQUIRE(heads % kv_heads == 0, "heads must be a multiple of kv_heads");
  IX_REQUIRE(ix_attention_diff_prefill_fits(head_dim, value_dim, page_size),
             "head_dim and value_dim must be 64 or 128, pages a multiple of 16");
  IX_REQUIRE(window >= 0 && keep_first >= 0, "window and keep_first must not be negative");
  const int64_t groups = static_cast<int64_t>(n_tiles) * heads;
  IX_REQUIRE(groups < (int64_t(1) << 31), "too many tiles for one launch");
  if (n_tiles == 0 || tokens == 0) return 0;
  int page_shift = -1;  // log2 of the page size if it is a power of two
  for (int b = 4; b < 31; ++b)
    if (page_size == (1 << b)) page_shift = b;
#define LAUNCH(NB, NBV)                                                                                                   \
  hipLaunchKernelGGL((attn_diff_prefill_kernel<NB, NBV>), dim3(static_cast<unsigned>(groups)), dim3(256), 0, stream,        \
                     (const __bf16*)q, (const __bf16*)k_cache, (const __bf16*)v_cache, block_table, tile_seq, tile_q0,       \
                     tile_rows, positions, (__bf16*)out, n_tiles, heads, kv_heads, page_size, max_blocks,                    \
                     scale * 1.4426950408889634f, window, keep_first, page_shift, lambda, eps, mult)
  if (head_dim == 64) {
    if (value_dim == 64) LAUNCH(4, 4);
    else LAUNCH(4, 8);
  } else {
    if (value_dim == 64) LAUNCH(8, 4);
    else LAUNCH(8, 8);
  }
#undef LAUNCH
  return ix_check_launch("ix_attention_diff_prefill");
}
