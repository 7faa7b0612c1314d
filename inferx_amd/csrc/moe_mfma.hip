// Grouped expert products on the matrix cores: bfloat16 in, float32 accumulate, or all of it float32 (template
// parameter TI; v_mfma_f32_16x16x4_f32, every product and sum in 32 bits).
//
//   GATE_UP: act[r, n] = silu(x[rows[r]] . W[e][n]) * (x[rows[r]] . W[e][N + n]),  W [E, 2N, K]
//   else:    y[r, n]   = a[r] . W[e][n],                                           W [E, N, K]
// for the rows r of expert e, taken from the row-tile map that the grouping
// kernel wrote (reference: GroupedGemmBf16Kernel, src/backends/cuda/ops/moe.cu:323-392,
// which uses scalar FMAs; SwiGLU src/model/moe_ffn.cc:288-291).
//
// The product is formed transposed, out^T[n][r] = W[n][:] . x[r][:], so that the
// big operand, the expert's weight rows, is the A operand and streams from
// memory straight into registers: v_mfma_f32_16x16x32_bf16, A = 16 weight rows,
// B = 16 activation rows, lane l of the result holding out-features 4*(l/16)+i
// of row l%16, i.e. four consecutive numbers of one output row.
//
// A wavefront owns 16 out-features x (16 * MT) rows.  Per iteration it covers
// 128 of K (in float32 64: 256 bytes of a row either way).  The matrix cores want
// 64 contiguous bytes of sixteen rows at once, memory wants whole lines of 128:
// so a load brings 128 contiguous bytes of eight weight rows, past the caches
// (non-temporal: a tile of rows uses a weight once), and the wavefront turns them over
// through 4 KB of LDS of its own, with no workgroup barrier.  The activations, which every
// workgroup reads, come from the caches as operands: in load j lane (m, g) reads
// the 16 bytes at k0 + 32 j + 8 g of row m (in float32 the j-th numbers of the four
// groups' pieces meet in one instruction).  KSPLIT = 4 (decoding: few rows, the
// weights are the traffic) lets the four wavefronts of a workgroup take a quarter
// of K each and add up through LDS; KSPLIT = 1 gives each wavefront its own 16
// out-features.
//
// What bounds it is the weights.  Against half lines straight into the operands' registers, through the caches, us (the
// same bits; non-temporal half lines are slower than either: a line's other half is gone when it is asked for):
// experts of 1,408 and a shared one of 5,632, rows of 2,048 numbers, both products: one row 16.3 + 10.9 (20.8 + 12.8), eight
// rows on 24 experts 49.5 + 25.8 (59.1 + 30.2; 6.5 TB/s), 32 rows on 43 experts 90 + 46 (106 + 56); experts of 2,560 and a
// shared one of 20,480, rows of 3,584, eight rows on 41 experts 264 + 130 (322 + 166).  The logits of a vocabulary of
// 151,936, rows of 2,048: one 95 (111), eight 98 (134), sixteen 110 (154), 32 153 (184); of 3,584: sixteen 197 (273).  Two
// blocks of weights a wavefront (gate|up, logits) take three wavefronts a SIMD, in whose registers nothing is spilled.
//
// Past the caches also where several tiles of sixteen rows ask for the same weights (steps of 17 to 48 rows, the shared
// expert's tiles): they are read again, and it is still faster than lines that stay (us, both products in turn at those sizes,
// past | through the caches: 17 rows 142 | 155, 32 162 | 175, 33 with the shared expert in pieces 162 | 176, 45 173 | 187).
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// 16 bytes of an operand, and what one of them against another adds to a 16 x 16 block of sums
template <typename TI> struct MfmaPiece;
template <> struct MfmaPiece<__bf16> {
  typedef bf16x8 type;
  static constexpr int N = 8;
  static __device__ __forceinline__ type zero() {
    return type{(__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f};
  }
  static __device__ __forceinline__ f32x4 mac(type w, type x, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, acc, 0, 0, 0);
  }
};
template <> struct MfmaPiece<float> {
  typedef f32x4 type;
  static constexpr int N = 4;
  static __device__ __forceinline__ type zero() { return type{0.f, 0.f, 0.f, 0.f}; }
  static __device__ __forceinline__ f32x4 mac(type w, type x, f32x4 acc) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], x[j], acc, 0, 0, 0);
    return acc;
  }
};

// LDS that a wavefront turns its weights over in, bytes: a round of each of its blocks of sixteen rows
#define IX_TURN_BYTES(NACC) (4096 * (NACC))

// The work of one wavefront (KSPLIT == 1) or workgroup (KSPLIT > 1): rows [row0, row_end) x out-features
// [n0, n0 + 16) of expert e.  `lds`: IX_TURN_BYTES for each wavefront; the partial sums of a split reduction go the same
// way.  NB: blocks of 16 out-features side by side ([n0, n0 + 16 NB)), so that the rows are read once for all of them.
// HALVES (up to eight rows, MT = NB = 1, width a multiple of two pieces): eight out-features; a block's second eight weight
// rows are the same features' second half of the reduction, and its second eight columns the rows' second halves, so that
// the sums meet on the diagonal of the 16 x 16 block and twice as many workgroups share few features.  Of a gated product
// (NB = 1) the second eight weight rows are the eight features' up rows, over the whole reduction and for any rows.
template <int MT, bool GATE_UP, int KSPLIT, typename TI, typename TO, int NB = 1, bool HALVES = false>
__device__ __forceinline__ void grouped_body(const TI* a, const TI* w,
                                             TO* __restrict__ out, const int32_t* __restrict__ rows, int e,
                                             int row0, int row_end, int n0, int n_out, int width, char* lds,
                                             int act = 0, float glu_limit = 0.f, const void* bias = nullptr,
                                             int bias_dtype = 0) {
  typedef MfmaPiece<TI> Piece;
  typedef typename Piece::type piece_t;
  constexpr int PN = Piece::N, ROUND = 16 * PN;  // numbers of a piece; of a round of four loads
  constexpr bool UP8 = HALVES && GATE_UP;
  constexpr int NACC = NB * (GATE_UP && !UP8 ? 2 : 1);  // accumulator b + NB h: block b of the gate (h = 0) or up (1) rows
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4;
  static_assert(!HALVES || (NB == 1 && (MT == 1 || GATE_UP)), "two halves of one block");
  const int span = HALVES && !GATE_UP ? width / 2 : width;  // the reduction as the matrix cores see it
  const int kper = KSPLIT > 1 ? (((span + KSPLIT - 1) / KSPLIT + ROUND - 1) & ~(ROUND - 1)) : span;
  const int kbegin = KSPLIT > 1 ? wave * kper : 0;
  const int kend = min(span, kbegin + kper);

  const int64_t w_rows = GATE_UP ? 2 * static_cast<int64_t>(n_out) : n_out;
  // In load j lane l reads piece 8 (j / 2) + l % 8 of row 8 (j % 2) + l / 8: whole lines of 128 bytes.  (A block's rows
  // start at an address that is the same for all lanes; beside it a lane counts pieces of 16 bytes: in bytes, row 15 of
  // 143 million numbers is past 32 bits.)
  const char* wbase[NACC];
  unsigned wrow[NB][2];
#pragma unroll
  for (int u = 0; u < NACC; ++u) {
    const int first = min(n0 + 16 * (u % NB), n_out - 1);  // (rows past the end: the last one, computed and not stored)
    wbase[u] = reinterpret_cast<const char*>(w + (static_cast<int64_t>(e) * w_rows + (u / NB) * static_cast<int64_t>(n_out) + first) * width);
    if (u < NB)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        wrow[u][h] = static_cast<unsigned>(min((HALVES ? 0 : 8 * h) + (lane >> 3), n_out - 1 - first)) * static_cast<unsigned>(width / PN) +
                     (HALVES && !GATE_UP && h ? span / PN : 0);
  }
  const char* const wup = UP8 ? wbase[0] + static_cast<int64_t>(n_out) * width * sizeof(TI) : nullptr;
  // Piece p of row r of a round lies at piece p ^ (r / 2 + 8 (r % 2)) of its 256 bytes: the rows that sixteen lanes read at
  // one piece, and the pieces of two rows that they write, fall on sixteen different groups of four banks.
  char* const turn = lds + wave * IX_TURN_BYTES(NACC);
  auto turn_at = [&](int r, int p) { return turn + 256 * r + 16 * (p ^ ((r >> 1) | ((r & 1) << 3))); };

  const TI* xr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int r = min(row0 + 16 * t + (HALVES && !GATE_UP ? m & 7 : m), row_end - 1);
    xr[t] = a + static_cast<int64_t>(rows ? rows[r] : r) * width + (HALVES && !GATE_UP && m >= 8 ? span : 0);
  }

  f32x4 acc[NACC][MT];
#pragma unroll
  for (int u = 0; u < NACC; ++u)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const piece_t zero = Piece::zero();
  // The loads of the next round of K are issued before the products of the present one, so that a wavefront
  // always has loads on their way.  Every load is unconditional (a piece past the end of a ragged last round is
  // read from the range's first piece instead, which is in the cache, and the activations' values are replaced
  // by zeros when they are used): with no branch in it the loop is one straight line, and the compiler lets the
  // younger loads stay in flight at each wait instead of waiting for all.
  piece_t fw[2][NACC][4], fx[2][MT][4];
  auto fetch = [&](int k0, piece_t (&w_)[NACC][4], piece_t (&x_)[MT][4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      int kk = k0 + PN * (4 * j + g);  // the four lane groups cover 64 contiguous bytes of a row per load
      kk = kk < kend ? kk : kbegin;  // (the range's first piece: it exists, kbegin + PN g need not)
      int kw = k0 + PN * (8 * (j >> 1) + (lane & 7));
      kw = kw < kend ? kw : kbegin;
#pragma unroll
      for (int u = 0; u < NACC; ++u)
        w_[u][j] = __builtin_nontemporal_load(
            reinterpret_cast<const piece_t*>(UP8 && (j & 1) ? wup : wbase[u]) + (wrow[u % NB][j & 1] + static_cast<unsigned>(kw) / PN));
#pragma unroll
      for (int t = 0; t < MT; ++t) x_[t][j] = *reinterpret_cast<const piece_t*>(xr[t] + kk);
    }
  };
  // (what the last round left is read before it is written over)
  auto turn_over = [&](piece_t (&w_)[NACC][4]) {
    ix_wave_lds_order();
#pragma unroll
    for (int u = 0; u < NACC; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<piece_t*>(turn_at(8 * (j & 1) + (lane >> 3), 8 * (j >> 1) + (lane & 7)) + 4096 * u) = w_[u][j];
    ix_wave_lds_order();
  };
  auto multiply = [&](int k0, const piece_t (&x_)[MT][4]) {
    piece_t w_[NACC][4];
#pragma unroll
    for (int u = 0; u < NACC; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) w_[u][j] = *reinterpret_cast<const piece_t*>(turn_at(m, 4 * j + g) + 4096 * u);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool ok = k0 + PN * (4 * j + g) < kend;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const piece_t xv = ok ? x_[t][j] : zero;
#pragma unroll
        for (int u = 0; u < NACC; ++u) acc[u][t] = Piece::mac(w_[u][j], xv, acc[u][t]);
      }
    }
  };
  // Rounds in pairs, so that the register sets are named statically; the loop runs while both rounds of a
  // turn are followed by another one and has no way out of its middle, the last one or two rounds come after it.
  const int rounds = kbegin < kend ? (kend - kbegin + ROUND - 1) / ROUND : 0;
  if (rounds > 0) {
    fetch(kbegin, fw[0], fx[0]);
    int k0 = kbegin, left = rounds;
    for (; left > 2; left -= 2, k0 += 2 * ROUND) {
      fetch(k0 + ROUND, fw[1], fx[1]);
      __builtin_amdgcn_sched_barrier(0);
      turn_over(fw[0]);
      multiply(k0, fx[0]);
      __builtin_amdgcn_sched_barrier(0);
      fetch(k0 + 2 * ROUND, fw[0], fx[0]);
      __builtin_amdgcn_sched_barrier(0);
      turn_over(fw[1]);
      multiply(k0 + ROUND, fx[1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (left == 2) {
      fetch(k0 + ROUND, fw[1], fx[1]);
      __builtin_amdgcn_sched_barrier(0);
      turn_over(fw[0]);
      multiply(k0, fx[0]);
      turn_over(fw[1]);
      multiply(k0 + ROUND, fx[1]);
    } else {
      turn_over(fw[0]);
      multiply(k0, fx[0]);
    }
  }

  if (KSPLIT > 1) {
    // the other wavefronts hand their partial sums to wavefront 0
    if (wave > 0) {
      float* dst = reinterpret_cast<float*>(turn) + lane * (MT * NACC * 4);
#pragma unroll
      for (int u = 0; u < NACC; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) dst[(u * MT + t) * 4 + i] = acc[u][t][i];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int s = 0; s < KSPLIT - 1; ++s) {
      const float* src = reinterpret_cast<const float*>(lds + (s + 1) * IX_TURN_BYTES(NACC)) + lane * (MT * NACC * 4);
#pragma unroll
      for (int u = 0; u < NACC; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[u][t][i] += src[(u * MT + t) * 4 + i];
    }
  }

  float ups[UP8 ? MT : 1][4];
  if constexpr (UP8) {  // lanes of the gate's rows: the up rows' sums are eight rows further on
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) ups[t][i] = __shfl_xor(acc[0][t][i], 32, 64);
    if (g >= 2) return;
  } else if constexpr (HALVES) {  // lanes of features and rows below eight: the other halves' sums are eight further on in both
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[0][0][i] += __shfl(acc[0][0][i], lane + 40, 64);
    if (m >= 8 || g >= 2) return;
  }
  // lane holds out-features n0 + 16 u + 4 g + i of row row0 + 16 t + m
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int nb = n0 + 16 * u + 4 * g;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int r = row0 + 16 * t + m;
      if (r >= row_end) continue;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = acc[u][t][i];
        const int c = min(nb + i, n_out - 1);
        if (bias) v[i] += ix_load_rt(bias, bias_dtype, c);
        if constexpr (GATE_UP) {
          float up = UP8 ? ups[UP8 ? t : 0][i] : acc[UP8 ? 0 : NB + u][t][i];
          if (bias) up += ix_load_rt(bias, bias_dtype, static_cast<int64_t>(n_out) + c);
          v[i] = ix_glu<sizeof(TI) == 2>(v[i], up, glu_limit);
        }
        if (!GATE_UP && act) v[i] = v[i] > 0.f ? v[i] * v[i] : 0.f;  // the square of relu
      }
      TO* dst = out + static_cast<int64_t>(r) * n_out + nb;
      if (nb + 4 <= n_out && (n_out & 3) == 0) {
        if constexpr (sizeof(TO) == 4) {
          *reinterpret_cast<f32x4*>(dst) = f32x4{v[0], v[1], v[2], v[3]};
        } else {
          bf16x4 o = {(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
          *reinterpret_cast<bf16x4*>(dst) = o;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nb + i < n_out) dst[i] = (TO)v[i];
      }
    }
  }
}

// x [rows <= 16 * MT, width] . w^T -> [rows, n_out], the products of a decoding step: 16 NB out-features a workgroup, the
// reduction split over its KSPLIT wavefronts.
template <int MT, bool GATE_UP, int KSPLIT, int NB, typename TI, typename TO, bool HALVES = false>
__global__ void __launch_bounds__(64 * KSPLIT, MT > 1 ? 1 : NB * (GATE_UP && !HALVES ? 2 : 1) > 1 ? 3 : 4)
linear_skinny_kernel(const TI* x, const TI* w, TO* __restrict__ out, const void* bias, int bias_dtype, int rows, int n_out,
                     int width, float glu_limit) {
  __shared__ __attribute__((aligned(16))) char lds[KSPLIT * IX_TURN_BYTES(NB * (GATE_UP && !HALVES ? 2 : 1))];
  grouped_body<MT, GATE_UP, KSPLIT, TI, TO, NB, HALVES>(x, w, out, nullptr, 0, 0, rows, blockIdx.x * (HALVES ? 8 : 16 * NB),
                                                        n_out, width, lds, 0, glu_limit, bias, bias_dtype);
}

// Two such products that do not need each other in one launch (bfloat16, rows <= 16): the first `blocks` workgroups one of them, gated or
// plain, the rest the other, a plain one.  HALVES, HALVES2: eight out-features a workgroup (see grouped_body).
template <bool GATE_UP, int KSPLIT, bool HALVES, bool HALVES2>
__global__ void __launch_bounds__(64 * KSPLIT, GATE_UP && !HALVES ? 3 : 4)
linear_skinny_pair_kernel(const __bf16* x, const __bf16* w, __bf16* __restrict__ out, const void* bias, int bias_dtype, int n_out, int width,
                          float glu_limit, int blocks, const __bf16* x2, const __bf16* w2, __bf16* __restrict__ out2, int n_out2,
                          int width2, int rows) {
  __shared__ __attribute__((aligned(16))) char lds[KSPLIT * IX_TURN_BYTES(GATE_UP && !HALVES ? 2 : 1)];
  const int at = blockIdx.x;
  if (at < blocks)
    grouped_body<1, GATE_UP, KSPLIT, __bf16, __bf16, 1, HALVES>(x, w, out, nullptr, 0, 0, rows, at * (HALVES ? 8 : 16), n_out, width, lds, 0,
                                                                glu_limit, bias, bias_dtype);
  else
    grouped_body<1, false, KSPLIT, __bf16, __bf16, 1, HALVES2>(x2, w2, out2, nullptr, 0, 0, rows, (at - blocks) * (HALVES2 ? 8 : 16), n_out2,
                                                               width2, lds);
}

template <int MT, bool GATE_UP, int KSPLIT, typename TI>
__global__ void __launch_bounds__(256, MT > 1 ? 1 : GATE_UP ? 3 : 4)
moe_grouped_mfma_kernel(const TI* a, const TI* w, TI* __restrict__ out,
                        const int32_t* __restrict__ offsets, const int32_t* __restrict__ rows,
                        const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_row0,
                        const int32_t* __restrict__ tile_info, int n_out, int width, int act, float glu_limit) {
  __shared__ __attribute__((aligned(16))) char lds[4 * IX_TURN_BYTES(GATE_UP ? 2 : 1)];
  if (static_cast<int>(blockIdx.y) >= tile_info[0]) return;
  const int e = tile_expert[blockIdx.y];
  const int n0 = (KSPLIT > 1 ? blockIdx.x : blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
  if (n0 >= n_out) return;  // whole wavefront (KSPLIT == 1) or whole workgroup
  grouped_body<MT, GATE_UP, KSPLIT, TI, TI>(a, w, out, rows, e, tile_row0[blockIdx.y], offsets[e + 1], n0, n_out, width, lds,
                                    act, glu_limit);
}

// Routed experts and the shared expert in one launch (decoding: every launch saved counts).  The first
// n16_s * shared_tiles workgroups serve the shared expert, which is one more "expert" over all `shared_rows`
// tokens with weights and sizes of its own (first, because its reduction may be the longer one and the last
// workgroups to start set the kernel's end); the rest serve the routed experts' row tiles.
template <int MT, bool GATE_UP, int NB, typename TI>
__global__ void __launch_bounds__(256, MT > 1 ? 1 : NB * (GATE_UP ? 2 : 1) > 1 ? 3 : 4)
moe_grouped_dual_kernel(const TI* a, const TI* w, TI* __restrict__ out,
                        const int32_t* __restrict__ offsets, const int32_t* __restrict__ rows,
                        const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_row0,
                        const int32_t* __restrict__ tile_info, int max_tiles, int n_out, int width,
                        const TI* a_s, const TI* w_s, TI* __restrict__ out_s,
                        int shared_rows, int n_out_s, int width_s, float glu_limit, float glu_limit_s) {
  __shared__ __attribute__((aligned(16))) char lds[4 * IX_TURN_BYTES(NB * (GATE_UP ? 2 : 1))];
  const int n16_s = (n_out_s + 16 * NB - 1) / (16 * NB);  // column blocks of 16 NB out-features
  const int shared_blocks = n16_s * ((shared_rows + 16 * MT - 1) / (16 * MT));
  int idx = blockIdx.x;
  if (idx < shared_blocks) {
    const int tile = idx / n16_s;
    grouped_body<MT, GATE_UP, 4, TI, TI, NB>(a_s, w_s, out_s, nullptr, 0, tile * 16 * MT, shared_rows,
                                             (idx - tile * n16_s) * 16 * NB,
                                 n_out_s, width_s, lds, 0, glu_limit_s);
  } else {
    idx -= shared_blocks;
    const int n16_e = (n_out + 16 * NB - 1) / (16 * NB);
    const int tile = idx / n16_e;
    if (tile >= tile_info[0]) return;
    const int e = tile_expert[tile];
    grouped_body<MT, GATE_UP, 4, TI, TI, NB>(a, w, out, rows, e, tile_row0[tile], offsets[e + 1],
                                             (idx - tile * n16_e) * 16 * NB, n_out, width, lds, 0, glu_limit);
  }
}

// `max_tiles` bounds the number of row tiles (the grid); the kernel reads the true number from tile_info.
// tile_rows (16, 32 or 64) must be what the grouping kernel was given.  gate_up: 0 a plain product, 1 gate|up rows
// with SwiGLU, 2 a plain product whose results pass the square of relu.  glu_limit > 0: the gate|up rows meet in
// the clamped form (`ix_glu`).  dtype: all of a, w and out (float32: tiles of 16 rows and k_split 4 only, which is what
// steps of few rows take).
#define IX_REQUIRE_PIECES(dtype, width)                                                                     \
  IX_REQUIRE(dtype == IX_F32 || dtype == IX_BF16, "dtype must be float32 or bfloat16");                      \
  IX_REQUIRE(width % (dtype == IX_F32 ? 4 : 8) == 0, "rows of the reduction must be multiples of 16 bytes")
extern "C" int ix_moe_grouped_mfma(const void* a, const void* w, void* out, int dtype, const int32_t* offsets,
                                   const int32_t* rows, const int32_t* tile_expert, const int32_t* tile_row0,
                                   const int32_t* tile_info, int max_tiles, int tile_rows, int64_t n_out,
                                   int64_t width, int gate_up, int k_split, float glu_limit, hipStream_t stream) {
  IX_REQUIRE(n_out > 0 && width > 0 && max_tiles >= 0, "sizes must be positive");
  IX_REQUIRE_PIECES(dtype, width);
  IX_REQUIRE(n_out < (1 << 30) && width < (1 << 30), "sizes too large");
  IX_REQUIRE(tile_rows == 16 || tile_rows == 32 || tile_rows == 64, "tile_rows must be 16, 32 or 64");
  IX_REQUIRE(k_split == 1 || k_split == 4, "k_split must be 1 or 4");
  IX_REQUIRE(dtype == IX_BF16 || (tile_rows == 16 && k_split == 4), "float32: tiles of 16 rows and k_split 4 only");
  IX_REQUIRE(gate_up >= 0 && gate_up <= 2, "gate_up must be 0, 1 or 2");
  IX_REQUIRE(max_tiles <= 65535, "too many row tiles for one launch");
  if (max_tiles == 0) return 0;
  const int n_tiles16 = static_cast<int>((n_out + 15) / 16);
  dim3 grid(k_split > 1 ? n_tiles16 : (n_tiles16 + 3) / 4, max_tiles), block(256);
#define LAUNCH(MT, GU, KS, TI)                                                                                    \
  hipLaunchKernelGGL((moe_grouped_mfma_kernel<MT, GU, KS, TI>), grid, block, 0, stream, (const TI*)a,             \
                     (const TI*)w, (TI*)out, offsets, rows, tile_expert, tile_row0, tile_info, (int)n_out,         \
                     (int)width, gate_up == 2 ? 1 : 0, glu_limit)
#define PICK(MT)                                       \
  if (gate_up == 1) {                                  \
    if (k_split > 1) LAUNCH(MT, true, 4, __bf16);      \
    else LAUNCH(MT, true, 1, __bf16);                  \
  } else {                                             \
    if (k_split > 1) LAUNCH(MT, false, 4, __bf16);     \
    else LAUNCH(MT, false, 1, __bf16);                 \
  }
  if (dtype == IX_F32) {
    if (gate_up == 1) LAUNCH(1, true, 4, float);
    else LAUNCH(1, false, 4, float);
  } else if (tile_rows == 16) { PICK(1) } else if (tile_rows == 32) { PICK(2) } else { PICK(4) }
#undef PICK
#undef LAUNCH
  return ix_check_launch("ix_moe_grouped_mfma");
}

// One launch for the routed experts (as ix_moe_grouped_mfma with k_split 4) and the shared expert
// (a_s [shared_rows, width_s] . w_s[(2) n_out_s, width_s]^T -> out_s [shared_rows, n_out_s]).
extern "C" int ix_moe_grouped_dual(const void* a, const void* w, void* out, int dtype, const int32_t* offsets,
                                   const int32_t* rows, const int32_t* tile_expert, const int32_t* tile_row0,
                                   const int32_t* tile_info, int max_tiles, int tile_rows, int64_t n_out,
                                   int64_t width, const void* a_s, const void* w_s, void* out_s, int shared_rows,
                                   int64_t n_out_s, int64_t width_s, int gate_up, float glu_limit, float glu_limit_s,
                                   hipStream_t stream) {
  IX_REQUIRE(n_out > 0 && width > 0 && n_out_s > 0 && width_s > 0 && max_tiles >= 0 && shared_rows > 0,
             "sizes must be positive");
  IX_REQUIRE_PIECES(dtype, width);
  IX_REQUIRE_PIECES(dtype, width_s);
  IX_REQUIRE(n_out < (1 << 24) && width < (1 << 30) && n_out_s < (1 << 24) && width_s < (1 << 30), "sizes too large");
  IX_REQUIRE(tile_rows == 16 || tile_rows == 32 || tile_rows == 64, "tile_rows must be 16, 32 or 64");
  IX_REQUIRE(dtype == IX_BF16 || tile_rows == 16, "float32: tiles of 16 rows only");
  // one column block per workgroup: two (the rows read once for 32 out-features) measured slower at every tile
  // height, 64 against 60 us for the gate|up product of a decoding step, for want of wavefronts in flight
  const int nb = 1;
  const int64_t n16_e = (n_out + 16 * nb - 1) / (16 * nb), n16_s = (n_out_s + 16 * nb - 1) / (16 * nb);
  const int64_t shared_tiles = (shared_rows + tile_rows - 1) / tile_rows;
  const int64_t blocks = n16_e * max_tiles + n16_s * shared_tiles;
  IX_REQUIRE(blocks < (1ll << 31), "too many workgroups");
  dim3 grid(static_cast<unsigned>(blocks)), block(256);
#define LAUNCH(MT, GU, NB, TI)                                                                                    \
  hipLaunchKernelGGL((moe_grouped_dual_kernel<MT, GU, NB, TI>), grid, block, 0, stream, (const TI*)a, (const TI*)w, \
                     (TI*)out, offsets, rows, tile_expert, tile_row0, tile_info, max_tiles, (int)n_out,            \
                     (int)width, (const TI*)a_s, (const TI*)w_s, (TI*)out_s, shared_rows, (int)n_out_s,             \
                     (int)width_s, glu_limit, glu_limit_s)
#define PICK(MT, NB)                          \
  if (gate_up == 1) LAUNCH(MT, true, NB, __bf16); \
  else LAUNCH(MT, false, NB, __bf16);
  if (dtype == IX_F32) {
    if (gate_up == 1) LAUNCH(1, true, 1, float);
    else LAUNCH(1, false, 1, float);
  } else if (tile_rows == 16) { PICK(1, 1) } else if (tile_rows == 32) { PICK(2, 1) } else { PICK(4, 1) }
#undef PICK
#undef LAUNCH
  return ix_check_launch("ix_moe_grouped_dual");
}

// out [rows, n_out] = x [rows, width] . w[n_out, width]^T, rows <= 64, operands of `dtype`; out of `dtype` or float32.
// gate_up 1: w is [2 n_out, width], gate rows and then up rows, which meet in the gated unit (`ix_glu` with glu_limit).
// `bias`: as many numbers as w has rows, added to the sums (to both before they meet), or null.
//
// What bounds it: the weights, and where they are few the launch itself and how many bytes a compute unit has on their
// way.  A product of the run's type is a workgroup of 16 out-features; with no more of them than the chip has compute
// units eight wavefronts split its reduction instead of four.  The float32 result (the logits) has so many out-features
// that 32 a workgroup are better: the rows, which every workgroup reads, weigh less beside the weights.
// Eight rows: 2,048 features of 2,048 numbers 4.9 us, of 5,632 9.6 (11.7 before whole lines were read), 11,264 features of
// 2,048 10.9 (14.6); a gated unit with biases saves the launch behind it, 6.2 us.  With eight features a workgroup (HALVES), one
// | eight rows, where sixteen took nine rows: 2,048 features of 2,048 3.7 | 4.3 (4.7), of 5,632 6.2 | 8.1 (9.1), 256 of 8,192
// 5.2 | 7.9 (10.0).
extern "C" int ix_linear_skinny(const void* x, const void* w, int dtype, void* out, int out_f32, const void* bias,
                                int bias_dtype, int rows, int64_t n_out, int64_t width, int gate_up, float glu_limit,
                                hipStream_t stream) {
  IX_REQUIRE(rows > 0 && rows <= 64 && n_out > 0 && width > 0, "between 1 and 64 rows, positive sizes");
  IX_REQUIRE_PIECES(dtype, width);
  IX_REQUIRE(n_out < (1ll << 31) - 32 && width < (1 << 30), "sizes too large");
  IX_REQUIRE(!out_f32 || !gate_up, "the gated unit's result is of the operands' type");
  const int per = out_f32 ? 32 : 16;
  const unsigned blocks = static_cast<unsigned>((n_out + per - 1) / per);
  const bool split8 = !out_f32 && blocks <= 256 && rows <= 32;
#define LAUNCH(MT, GU, KS, NB, TI, TO)                                                                                      \
  hipLaunchKernelGGL((linear_skinny_kernel<MT, GU, KS, NB, TI, TO>), dim3(blocks), dim3(64 * KS), 0, stream, (const TI*)x, \
                     (const TI*)w, (TO*)out, bias, bias_dtype, rows, (int)n_out, (int)width, glu_limit)
#define BY_FORM(MT, KS, TI)                        \
  if (gate_up) LAUNCH(MT, true, KS, 1, TI, TI);    \
  else LAUNCH(MT, false, KS, 1, TI, TI)
#define BY_ROWS(TI)                                      \
  if (split8 && rows <= 16) { BY_FORM(1, 8, TI); }       \
  else if (split8) { BY_FORM(2, 8, TI); }                \
  else if (rows <= 16) { BY_FORM(1, 4, TI); }            \
  else if (rows <= 32) { BY_FORM(2, 4, TI); }            \
  else { BY_FORM(4, 4, TI); }
#define LOGITS(TI)                                              \
  if (rows <= 16) LAUNCH(1, false, 4, 2, TI, float);            \
  else if (rows <= 32) LAUNCH(2, false, 4, 2, TI, float);       \
  else LAUNCH(4, false, 4, 2, TI, float)
  // Few features for few rows: eight of them a workgroup where sixteen leave half the compute units without one.  (bfloat16
  // only: float32 rows are then summed up in another order in portions of up to eight rows than in longer ones, and two
  // scores of a router 1.8e-6 apart fell the other way from the 64-bit result.)
  if (dtype == IX_BF16 && !out_f32 && !gate_up && rows <= 8 && blocks <= 128 && width % 16 == 0) {
    hipLaunchKernelGGL((linear_skinny_kernel<1, false, 8, 1, __bf16, __bf16, true>), dim3(static_cast<unsigned>((n_out + 7) / 8)),
                       dim3(512), 0, stream, (const __bf16*)x, (const __bf16*)w, (__bf16*)out, bias, bias_dtype, rows,
                       (int)n_out, (int)width, glu_limit);
    return ix_check_launch("ix_linear_skinny");
  }
  // A gated product with more than one and at most one and a half blocks of sixteen for each of the 256 compute units: some have
  // two of them and most one; of eights each has up to three.  One | eight rows of 2,048 numbers, us, sixteens and eights,
  // bfloat16: 257 blocks 9.4 | 10.5 and 8.5 | 9.6, 320 10.2 | 11.0 and 9.1 | 10.1, 384 10.3 | 11.2 and 9.7 | 10.4; with a fourth
  // eight for some 416 10.6 | 11.5 and 11.3 | 12.5.  float32: 257 18.9 | 19.8 and 16.0 | 17.2, 384 20.5 | 21.2 and 17.9 | 19.1, 416
  // 20.5 | 21.4 and 21.2 | 23.1.
  if (!out_f32 && gate_up && rows <= 8 && blocks > 256 && blocks <= 384) {
    const dim3 grid8(static_cast<unsigned>((n_out + 7) / 8));
    if (dtype == IX_F32)
      hipLaunchKernelGGL((linear_skinny_kernel<1, true, 4, 1, float, float, true>), grid8, dim3(256), 0, stream, (const float*)x,
                         (const float*)w, (float*)out, bias, bias_dtype, rows, (int)n_out, (int)width, glu_limit);
    else
      hipLaunchKernelGGL((linear_skinny_kernel<1, true, 4, 1, __bf16, __bf16, true>), grid8, dim3(256), 0, stream, (const __bf16*)x,
                         (const __bf16*)w, (__bf16*)out, bias, bias_dtype, rows, (int)n_out, (int)width, glu_limit);
    return ix_check_launch("ix_linear_skinny");
  }
  if (out_f32 && dtype == IX_F32) { LOGITS(float); }
  else if (out_f32) { LOGITS(__bf16); }
  else if (dtype == IX_F32) { BY_ROWS(float) }
  else { BY_ROWS(__bf16) }
#undef LOGITS
#undef BY_ROWS
#undef BY_FORM
#undef LAUNCH
  return ix_check_launch("ix_linear_skinny");
}

// Two products of the same few rows' layer that do not need each other, in one launch: out [rows, n_out] = x . w^T as ix_linear_skinny
// forms it (gate_up, bias, glu_limit) and out2 [rows, n_out2] = x2 [rows, width2] . w2^T, all bfloat16, up to 16 rows.
//
// What it saves is a launch's start and its first loads' way from memory, during which the other product's weights arrive: never slower
// than two launches (one, eight and sixteen rows, 19 pairs of 768 to 14,336 features of 768 to 18,944 numbers, weights from memory).
// Eights or sixteens, us, one | eight rows, two launches / sixteens / eights:
//   gated, up to 600 blocks of sixteen together: 88 + 228 of 2,048 numbers 10.7 / 7.6 / 6.7 | 11.9 / 8.7 / 7.4, 176 + 384 14.6 / 11.2 /
//   10.3 | 16.3 / 11.9 / 10.4, 352 + 228 15.6 / 13.4 / 12.5 | 16.8 / 13.8 / 12.8; more: 256 + 384 16.7 / 11.7 / 11.9 | 17.8 / 12.5 / 12.6,
//   384 + 384 18.0 / 14.9 / 14.8 | 19.8 / 14.4 / 15.3, 352 + 640 21.0 / 16.9 / 17.1 | 22.4 / 17.3 / 17.7
//   plain, up to 128 blocks each, as alone: 128 of 5,632 and 128 of 2,048 numbers 9.9 / 8.4 / 7.3 | 11.8 / 9.5 / 9.2, of 11,264 13.6 / 13.5 /
//   10.8 | 17.5 / 15.8 / 14.0; more: 224 of 18,944 and 224 of 3,584 32.5 / 30.1 / 28.5 | 37.2 / 32.5 / 38.0, 256 of 11,008 and 256 of
//   4,096 26.2 / 22.7 / 24.7 | 28.5 / 24.5 / 32.1
extern "C" int ix_linear_skinny_pair(const void* x, const void* w, void* out, const void* bias, int bias_dtype, int64_t n_out,
                                     int64_t width, int gate_up, float glu_limit, const void* x2, const void* w2, void* out2,
                                     int64_t n_out2, int64_t width2, int rows, hipStream_t stream) {
  IX_REQUIRE(rows > 0 && rows <= 16 && n_out > 0 && width > 0 && n_out2 > 0 && width2 > 0, "between 1 and 16 rows, positive sizes");
  IX_REQUIRE(width % 8 == 0 && width2 % 8 == 0, "rows of the reduction must be multiples of 16 bytes");
  IX_REQUIRE(n_out < (1 << 24) && n_out2 < (1 << 24) && width < (1 << 30) && width2 < (1 << 30), "sizes too large");
  const int64_t sixteens = (n_out + 15) / 16, sixteens2 = (n_out2 + 15) / 16;
  const bool eights = rows <= 8 && (gate_up ? sixteens + sixteens2 <= 600
                                            : sixteens <= 128 && sixteens2 <= 128 && width % 16 == 0 && width2 % 16 == 0);
  const int per = eights ? 8 : 16, per2 = eights && !gate_up ? 8 : 16;
  const int blocks = static_cast<int>((n_out + per - 1) / per), blocks2 = static_cast<int>((n_out2 + per2 - 1) / per2);
#define LAUNCH(GU, KS, H, H2)                                                                                                    \
  hipLaunchKernelGGL((linear_skinny_pair_kernel<GU, KS, H, H2>), dim3(static_cast<unsigned>(blocks + blocks2)), dim3(64 * KS), 0,   \
                     stream, (const __bf16*)x, (const __bf16*)w, (__bf16*)out, bias, bias_dtype, (int)n_out, (int)width, glu_limit, \
                     blocks, (const __bf16*)x2, (const __bf16*)w2, (__bf16*)out2, (int)n_out2, (int)width2, rows)
  if (gate_up) {
    if (eights) LAUNCH(true, 4, true, false);
    else LAUNCH(true, 4, false, false);
  } else {
    if (eights) LAUNCH(false, 8, true, true);
    else LAUNCH(false, 8, false, false);
  }
#undef LAUNCH
  return ix_check_launch("ix_linear_skinny_pair");
}
