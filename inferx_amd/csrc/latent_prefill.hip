// Attention over the compressed cache (see latent_attention.hip) for steps that bring requests many tokens, on the matrix
// cores: bfloat16; rank + rot_dim a multiple of 32 up to 576, rank a multiple of 16 up to 512.
//
// All heads read the same cached rows, so a workgroup of four wavefronts shares them through LDS, 32 keys a round:
//
//     S^T[key][column] = K[key][:] . Q[column][:]             (A = key rows, B = the column's query, in registers)
//     O^T[d][column]  += C^T[d][key] P^T[key][column]          (A = latent rows read transposed, B = the weights)
//
// v_mfma_f32_16x16x32_bf16 leaves lane l with column l % 16 and rows 4 (l / 16) + i.  Row m of the first 16 keys of a
// round is key 8 (m / 4) + m % 4, of the second key 8 (m / 4) + 4 + m % 4, so a lane holds the scores of keys
// 8 (l / 16) .. + 7 of its column: the B operand of the second product as it stands.  Softmax online, float32, per column.
//
// What bounds it: the LDS.  A wavefront that takes sixteen columns through both products reads an operand from LDS for
// every product, and writing the rows once more transposed takes as long again.  So each of a workgroup's four wavefronts
// works the scores of sixteen columns (a head's sixteen rows), leaves the weights in LDS, and then takes a quarter of the
// latent's numbers for all sixty-four columns: 48 operands read for 68 products, and registers for two wavefronts a SIMD,
// so that another workgroup's products cover this one's barriers.  The latent rows are transposed on the way out of LDS
// (ds_read_b64_tr_b16: of sixteen lanes, lanes 4 e .. 4 e + 3 name sixteen numbers of key e, and lane i gets the i-th
// number of the four keys).  Rows go from memory into LDS without passing registers, the next round's while this one is
// worked, in two buffers.
//
// A workgroup takes sixteen consecutive rows of the step and four heads.  Rows of several requests in a tile are worked
// request by request (the other rows' keys all masked: they change nothing).
//
// There are three forms by the size of a row; the smaller ones take less LDS, and more workgroups share a compute unit.
//
// Measured with 16 heads, one prompt of 2,048 tokens | 32 prompts of 160, us, against a head's sixteen columns in one
// wavefront through both products and the rows written transposed (latent + rotated numbers): 512 + 64 148 | 72 (378 | 145),
// 448 + 64 155 | 73 (353 | 137), 256 + 64 118 | 46 (216 | 88), 128 + 64 112 | 39 (163 | 69), 64 + 32 85 | 22 (109 | 25),
// 32 + 32 85 | 20.5 (86 | 21).  One form of 78 KB of LDS for all sizes took 113 | 35 and 111 | 33 us at the last two;
// branches past the products that a smaller row does without, 258 | 104 us at 448 + 64.
// With masks only where a column needs one, and no exchange between a column's lanes unless its maximum has outgrown the
// reference point: 512 + 64 140 (157 beside it), 256 + 64 104 (119), 128 + 64 98 (113), 64 + 32 71 (86) for 2,048 tokens.
#include "common.h"

typedef __bf16 lp_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 lp_bf16x4 __attribute__((ext_vector_type(4)));
typedef float lp_f32x4 __attribute__((ext_vector_type(4)));

#define LP_KEYS 32
// A row's numbers in LDS, by the size of the form: its first 16, 32 or 64 pieces of 16 bytes, and where there are more (at
// most eight) the rest in rows of their own.
constexpr int lp_main(int nw) { return nw <= 4 ? 128 : nw <= 10 ? 256 : 512; }
constexpr int lp_tail(int nw) { return 32 * nw > lp_main(nw) ? 64 : 0; }
constexpr int lp_lds_bytes(int nw) { return 256 + 2 * LP_KEYS * (64 + 2 * (lp_main(nw) + lp_tail(nw))); }
constexpr int lp_per_unit(int nw) { return nw <= 4 ? 4 : 2; }  // workgroups that a compute unit holds

// Where piece p of key row r lies among the rows' first pieces (or among their last eight): a row's pieces are permuted
// so that the sixteen rows that one product reads at one piece (8 a + b, or 8 a + 4 + b; a, b < 4) fall on all banks.
// One instruction fills 64 pieces in the order of the lanes (one, two or four rows), so it is the lanes' source
// addresses that are permuted.
__device__ __forceinline__ int lp_swap(int r) { return ((r >> 3) << 2) | (r & 3); }
__device__ __forceinline__ int lp_swap_tail(int r) { return ((r >> 3) << 1) | ((r >> 1) & 1); }
// 16 bytes of every live lane from memory into LDS, side by side in the order of the lanes
__device__ __forceinline__ void lp_bring(const __bf16* from, __bf16* to) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                   (__attribute__((address_space(3))) void*)to, 16, 0, 0);
}

typedef short lp_s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ lp_s16x4 lp_read_turned(const __bf16* at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lp_s16x4*)at);
}

// rank + rot_dim <= 32 NW, rank <= 16 NR.  The loops over a row always run to these sizes (behind a smaller row lie zeros):
// with a branch at each product the compiler waits for every operand.  FULL: both are these sizes, which are then numbers
// that the compiler knows (148 us instead of 157 at 2,048 tokens of 512 + 64, the largest form and the usual latent).
template <int NW, int NR, bool FULL>
__global__ void __launch_bounds__(256, lp_per_unit(NW))
latent_prefill_kernel(const __bf16* __restrict__ ql, int64_t ql_t, int64_t ql_h, const __bf16* __restrict__ qr,
                      int64_t qr_t, int64_t qr_h, const __bf16* __restrict__ cache,
                      const int32_t* __restrict__ block_table, const int32_t* __restrict__ seq_of_token,
                      const int32_t* __restrict__ positions, __bf16* __restrict__ out, int64_t out_t, int64_t out_h,
                      int tokens, int heads, int rank, int rot_dim, int page_size, int max_blocks, float scale_log2,
                      int n_tiles, int inwards, int window, const __bf16* __restrict__ head_gate, int64_t gate_stride) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lp_lds[];
  constexpr int DT = NR / 4;  // tiles of sixteen numbers of the latent that a wavefront sums up
  constexpr int MAIN = lp_main(NW), TAIL = lp_tail(NW);
  constexpr int PIECES = MAIN / 8, TOGETHER = 64 / PIECES;  // rows that one instruction brings
  const int width = FULL ? 32 * NW : rank + rot_dim;
  if (FULL) rank = 16 * NR;
  const int p8 = width / 8, nw = width / 32, nr = rank / 16;
  float* const alpha_s = reinterpret_cast<float*>(lp_lds);             // [4][16]: the factor of a column's sums; at the end 1 / sum
  __bf16* const p_s = reinterpret_cast<__bf16*>(alpha_s + 64);         // [4][16][32]: weights
  __bf16* const k_s = p_s + 4 * 16 * LP_KEYS;  // two buffers of rows: [32][MAIN], then [32][TAIL]
  constexpr int BUFFER = LP_KEYS * (MAIN + TAIL);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  // one row of workgroups, a tile's groups of four heads side by side; the tiles with the most keys first, or (inwards:
  // all workgroups are resident at once) the second half of them in the order of rising length,
  // so that a compute unit gets a long and a short one
  const int head_groups = (heads + 3) / 4;
  const int at = static_cast<int>(blockIdx.x) / head_groups, half = (n_tiles + 1) / 2;
  const int tile = (inwards && at >= half) ? at - half : n_tiles - 1 - at;
  const int r0 = tile * 16, r1 = min(r0 + 16, tokens), row = r0 + n;
  const int head0 = (static_cast<int>(blockIdx.x) % head_groups) * 4, head = head0 + wave;
  const int live_heads = min(4, heads - head0);
  const bool wave_on = head < heads, col_ok = wave_on && row < r1;

  lp_bf16x8 qf[NW];
#pragma unroll
  for (int s = 0; s < NW; ++s) {
#pragma unroll
    for (int e = 0; e < 8; ++e) qf[s][e] = static_cast<__bf16>(0.f);
    if ((FULL || s < nw) && col_ok) {
      const int i = 32 * s + 8 * g;
      const __bf16* src = i < rank ? ql + row * ql_t + head * ql_h + i : qr + row * qr_t + head * qr_h + (i - rank);
      qf[s] = *reinterpret_cast<const lp_bf16x8*>(src);
    }
  }
  lp_f32x4 acc[4][DT];  // [column group][tile of the latent]
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[c][d] = lp_f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -1e30f, l = 0.f;
  if (!FULL && width < 32 * NW) {  // (what no row fills is zero; the barrier before the first rows orders these writes)
    const lp_bf16x8 zero = {(__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f};
    for (int i = tid; i < 2 * BUFFER / 8; i += 256) *reinterpret_cast<lp_bf16x8*>(k_s + 8 * i) = zero;
  }

  int seg = r0;
  while (seg < r1) {  // (every decision in this loop is the same for the whole workgroup)
    const int seq = seq_of_token[seg];
    int end = seg + 1;
    while (end < r1 && seq_of_token[end] == seq) ++end;
    const int k_end = positions[end - 1] + 1;  // a request's rows come in the order of their positions
    // with a window W the first of these rows reads from key k_lo on, and no row reads an earlier one (whose page
    // may be gone); rounds start at multiples of their length
    const int k_lo = window > 0 ? max(positions[seg] + 1 - window, 0) : 0;
    const int k_begin = k_lo & ~(LP_KEYS - 1);
    const int my_pos = (col_ok && row >= seg && row < end) ? positions[row] : -1;
    const int my_lo = window > 0 ? my_pos - window : -1;  // the last key that this column does not read
    const int32_t* table = block_table + static_cast<int64_t>(seq) * max_blocks;

    // A wavefront brings eight keys of a round.  Keys that nobody reads are replaced by the nearest that somebody does.
    auto bring = [&](int k0, __bf16* to, int lane) {
      const int j0 = k0 + 8 * wave;
      const bool together = (page_size & 7) == 0 && j0 >= k_lo && j0 + 8 <= k_end;  // eight rows of one page
      const int64_t at0 = together ? (static_cast<int64_t>(table[j0 / page_size]) * page_size + j0 % page_size) * width : 0;
      auto row_at = [&](int u) {
        if (together) return at0 + u * width;
        const int j = max(min(j0 + u, k_end - 1), k_lo);
        return (static_cast<int64_t>(table[j / page_size]) * page_size + j % page_size) * width;
      };
#pragma unroll
      for (int u = 0; u < 8; u += TOGETHER) {
        const int v = TOGETHER > 1 ? u + lane / PIECES : u, r = 8 * wave + v, piece = (lane % PIECES) ^ lp_swap(r);
        const int64_t from = row_at(v);
        if (FULL || piece < p8) lp_bring(cache + from + 8 * piece, to + (8 * wave + u) * MAIN);
      }
      if constexpr (TAIL > 0) {
        const int r = 8 * wave + (lane >> 3), piece = PIECES + ((lane & 7) ^ lp_swap_tail(r));
        if (piece < p8) lp_bring(cache + row_at(lane >> 3) + 8 * piece, to + LP_KEYS * MAIN + 8 * wave * TAIL);
      }
    };
    __syncthreads();  // (the request before: its last round has been read)
    if (k_begin < k_end) bring(k_begin, k_s, lane);
    int buf = 0;
    for (int k0 = k_begin; k0 < k_end; k0 += LP_KEYS, buf ^= 1) {
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wavefront's rows are in LDS
      __syncthreads();                     // ... and everybody's; the round before has been read
      // The lane's number is hidden from the optimiser once a round: it would otherwise work out every place of the
      // permuted pieces before the loop and keep some forty registers for them, which are not there.
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int n_ = ln & 15, g_ = ln >> 4;
      const __bf16* rows = k_s + buf * BUFFER;
      if (k0 + LP_KEYS < k_end) bring(k0 + LP_KEYS, k_s + (buf ^ 1) * BUFFER, ln);
      __builtin_amdgcn_sched_barrier(0);
      if (wave_on) {
        lp_f32x4 s0 = lp_f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
        // key rows 8 a + b and, four rows on, 8 a + 4 + b: the same permutation, which acts on the last four bits of a
        // piece's number (a tail's on the last three), so pieces 4 q + g of q = i, i + 4, .. are a constant apart
        const int r = 8 * (n_ >> 2) + (n_ & 3);
        const __bf16* main_at[4];
        const __bf16* tail_at[2];  // (not used where there are none)
#pragma unroll
        for (int i = 0; i < 4; ++i) main_at[i] = rows + r * MAIN + (((4 * i + g_) ^ lp_swap(r)) << 3);
#pragma unroll
        for (int i = 0; i < 2; ++i) tail_at[i] = rows + LP_KEYS * MAIN + r * TAIL + (((4 * i + g_) ^ lp_swap_tail(r)) << 3);
        // (two pairs of operands on their way while one is multiplied; left to itself the compiler waits for every pair)
        lp_bf16x8 a0[3], a1[3];
        auto read = [&](int q) {
          const __bf16* at = q < MAIN / 32 ? main_at[q & 3] + 128 * (q >> 2) : tail_at[q & 1];
          a0[q % 3] = *reinterpret_cast<const lp_bf16x8*>(at);
          a1[q % 3] = *reinterpret_cast<const lp_bf16x8*>(at + 4 * (q < MAIN / 32 ? MAIN : TAIL));
        };
        read(0);
        read(1);
#pragma unroll
        for (int q = 0; q < NW; ++q) {
          if (q + 2 < NW) read(q + 2);
          __builtin_amdgcn_sched_barrier(0);
          s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[q % 3], qf[q], s0, 0, 0, 0);
          s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[q % 3], qf[q], s1, 0, 0, 0);
        }
        float p[8], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; ++i) p[i] = (i < 4 ? s0[i & 3] : s1[i & 3]) * scale_log2;
        if (!__all(k0 + LP_KEYS - 1 <= my_pos && k0 > my_lo)) {  // (rounds that every column sees need no mask)
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int j = k0 + 8 * g + i;
            p[i] = (j <= my_pos && j > my_lo) ? p[i] : -INFINITY;
          }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = fmaxf(mx, p[i]);
        // The reference point m of the exponentials follows the running maximum lazily: a column's moves only when its
        // maximum has outgrown it by more than 2^8, so the sums are seldom rescaled, and whether any has needs no exchange
        // between a column's four lanes.  Any m gives the same quotient; weights up to 2^8 keep the relative precision of
        // bfloat16.
        float alpha = 1.0f;
        if (__any(mx > m + 8.f)) {
          mx = fmaxf(mx, __shfl_xor(mx, 16));
          mx = fmaxf(mx, __shfl_xor(mx, 32));
          if (mx > m + 8.f) {
            alpha = exp2f(m - mx);
            m = mx;
            l *= alpha;
          }
        }
        lp_bf16x8 pb;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float w = __builtin_amdgcn_exp2f(p[i] - m);  // (v_exp_f32 as it is: a result below the smallest normal number may be 0)
          l += w;
          pb[i] = static_cast<__bf16>(w);
        }
        *reinterpret_cast<lp_bf16x8*>(p_s + ((wave * 16 + n) * 4 + g) * 8) = pb;
        if (g == 0) alpha_s[wave * 16 + n] = alpha;
      }
      // (not __syncthreads, which would also wait for the next round's rows: the weights and factors are all that is
      // handed over here)
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      float alpha[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) alpha[c] = alpha_s[c * 16 + n_];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (c >= live_heads || !__any(alpha[c] != 1.0f)) continue;
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[c][d] *= alpha[c];
      }
      lp_bf16x8 pb[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) pb[c] = *reinterpret_cast<const lp_bf16x8*>(p_s + ((c * 16 + n) * 4 + g) * 8);
      // this lane's part of the transposed reads: key 8 g + n / 4 (and four keys on), numbers 4 (n % 4) .. of a tile's
      // sixteen; they lie in piece 2 D + (n % 4) / 2 of the row (D the tile), and D and D + 8 are a constant apart
      const int r = 8 * g_ + (n_ >> 2), in_piece = 4 * (n_ & 1);
      const __bf16* at = rows + r * MAIN + in_piece;
      lp_s16x4 lo[2], hi[2];
      auto read = [&](int d) {
        const __bf16* from = at + (((2 * (wave * DT + d) + ((n_ >> 1) & 1)) ^ lp_swap(r)) << 3);
        lo[d & 1] = lp_read_turned(from);
        hi[d & 1] = lp_read_turned(from + 4 * MAIN);
      };
      read(0);
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        if (d + 1 < DT) read(d + 1);
        __builtin_amdgcn_sched_barrier(0);
        const lp_bf16x8 a = __builtin_bit_cast(lp_bf16x8, __builtin_shufflevector(lo[d & 1], hi[d & 1], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[c], acc[c][d], 0, 0, 0);
      }
    }
    seg = end;
  }

  float lt = l + __shfl_xor(l, 16);
  lt += __shfl_xor(lt, 32);
  __syncthreads();
  if (wave_on && g == 0)
    alpha_s[wave * 16 + n] = (head_gate && col_ok)
        ? 1.0f / (lt * (1.0f + __expf(-(float)head_gate[row * gate_stride + head]))) : 1.0f / lt;
  __syncthreads();
  if (row >= r1) return;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (c >= live_heads) continue;
    const float inv = alpha_s[c * 16 + n];
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      if (FULL || wave * DT + d < nr) {
        lp_bf16x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = static_cast<__bf16>(acc[c][d][i] * inv);
        *reinterpret_cast<lp_bf16x4*>(out + row * out_t + (head0 + c) * out_h + 16 * (wave * DT + d) + 4 * g) = o;
      }
    }
  }
}

// What ix_latent_attention_mfma does for steps that are not one token per request (it has checked the operands).
int ix_latent_prefill(const void* ql, int64_t ql_t, int64_t ql_h, const void* qr, int64_t qr_t, int64_t qr_h,
                      const void* cache, const int32_t* block_table, const int32_t* seq_of_token, const int32_t* positions,
                      void* out, int64_t out_t, int64_t out_h, int tokens, int heads, int rank, int rot_dim, int page_size,
                      int max_blocks, float scale_log2, int window, const void* head_gate, int64_t gate_stride,
                      hipStream_t stream) {
  const int width = rank + rot_dim, n_tiles = (tokens + 15) / 16;
  const int64_t groups = static_cast<int64_t>(n_tiles) * ((heads + 3) / 4);
  IX_REQUIRE(groups < (int64_t(1) << 31), "too many workgroups for one launch");
  const dim3 grid(static_cast<unsigned>(groups));
#define LAUNCH(NW, NR, FULL)                                                                                            \
  do {                                                                                                                  \
    auto kernel = latent_prefill_kernel<NW, NR, FULL>;                                                                  \
    constexpr size_t lds = lp_lds_bytes(NW);                                                                            \
    const int inwards = groups <= 256 * lp_per_unit(NW); /* (all of them on the 256 compute units at once) */           \
    if (lds > 48 * 1024) {                                                                                              \
      static bool raised = false;                                                                                       \
      if (!raised) {                                                                                                    \
        /* (a refusal shows as the launch's own error) */                                                              \
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,    \
                                  96 * 1024);                                                                           \
        (void)hipGetLastError();                                                                                        \
        raised = true;                                                                                                  \
      }                                                                                                                 \
    }                                                                                                                   \
    hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, (const __bf16*)ql, ql_t, ql_h, (const __bf16*)qr, qr_t,     \
                       qr_h, (const __bf16*)cache, block_table, seq_of_token, positions, (__bf16*)out, out_t, out_h,     \
                       tokens, heads, rank, rot_dim, page_size, max_blocks, scale_log2, n_tiles, inwards, window,       \
                       (const __bf16*)head_gate, gate_stride);                                                          \
  } while (0)
  if (width <= 128) LAUNCH(4, 8, false);
  else if (width <= 320 && rank <= 256) LAUNCH(10, 16, false);
  else if (width == 576 && rank == 512) LAUNCH(18, 32, true);
  else LAUNCH(18, 32, false);
#undef LAUNCH
  return ix_check_launch("ix_latent_attention_mfma");
}
