// Grouped expert products in float32 for more than a few rows per expert (prompt portions of a float32 run): operands
// staged through LDS, v_mfma_f32_16x16x4_f32, every product and sum in 32 bits.
//
// What bounds it: at a few dozen rows per expert the weights' way from memory, from about fifty on the matrix cores
// (32 cycles for 16 x 16 x 4).  A workgroup owns up to 64 rows of one expert (a tile of the grouping kernel's map: with
// a few hundred tokens all rows of an expert, so that its weights are read once) x 64 weight rows, which for gate|up are
// 32 gate rows and their 32 up rows; its four wavefronts take sixteen weight rows each (for gate|up eight and eight)
// and all of the tile's rows.  Stages of 32 of the reduction (128 bytes a row) go through two LDS buffers, three more
// are on their way in registers, one barrier a stage; 32 KB of LDS and 128 registers leave four workgroups to a compute
// unit, whose loads and products overlap.  Rows of LDS keep their eight 16-byte pieces permuted (piece p of row r at
// p ^ ((r >> 1) & 7)), so that sixteen rows read at one piece fall on different banks.
//
// A lane reads four consecutive numbers of its row at a time; product j of a piece multiplies the j-th of them, so the
// four slots of the reduction that one matrix instruction adds up are the pieces' j-th numbers, the same in both
// operands.  Workgroups start the reduction at a stage that follows from their column block and wrap round: rows of a
// power of two bytes would otherwise all ask the same memory channels at once.  The order of a result's sum so depends
// on its column alone.
//
// Measured at 511 tokens of 60 experts of 1,408 on a width of 2,048, 4 a token (34 rows an expert, 2.1 GB of weights):
// 387 + 195 us for the two products, against 805 + 563 us of the plain kernel (a workgroup of 64 x 64 on the vector
// units, LDS filled a number at a time).  The weights alone take 325 us at the rate of a pure read, the products 230.
// With the tiles cut evenly over the dies, routing to weighted sum: 361 tokens 502 -> 458 us, 511 591 -> 561, 800 797 -> 731.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define TF_ROWS 64                 // rows of a tile of the map
#define TF_WROWS 64                // weight rows per workgroup
#define TF_K 32                    // numbers of the reduction per stage
#define TF_TILE (TF_ROWS * TF_K)   // numbers of one LDS buffer
__device__ __forceinline__ int tf_at(int row, int piece) { return row * TF_K + ((piece ^ ((row >> 1) & 7)) << 2); }

// NT: sixteens of rows that the tile holds.  Every load is unconditional and the loop one straight line (see
// moe_tiled.hip): a stage past the end asks for the last stage again, a piece past the row's end for the row's start,
// with zeros written over it in LDS.
template <bool GATE_UP, int NT>
__device__ __forceinline__ void tiled_f32_body(const float* a, const float* w, float* out,
                                               const int32_t* __restrict__ rows, int n_out, int width, int e, int row0,
                                               int row_end, int col_block, float* ws, float* xs, int act,
                                               float glu_limit) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  constexpr int COLS = GATE_UP ? TF_WROWS / 2 : TF_WROWS;
  constexpr int NPX = (NT + 1) / 2;  // pieces of activations per thread and stage (32 rows at a time)
  const int n0 = col_block * COLS;

  const int64_t w_rows = GATE_UP ? 2 * static_cast<int64_t>(n_out) : n_out;
  const float* w_expert = w + static_cast<int64_t>(e) * w_rows * width;
  const int kc_mine = (tid & 7) * 4;
  int wsrc[2], xsrc[NPX];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (tid >> 3) + 32 * i;  // LDS row; wavefront r / 16 multiplies it
    const int src = GATE_UP ? ((r & 8) ? n_out : 0) + min(n0 + 8 * (r >> 4) + (r & 7), n_out - 1) : min(n0 + r, n_out - 1);
    wsrc[i] = src * width;
  }
#pragma unroll
  for (int i = 0; i < NPX; ++i) {
    const int gr = min(row0 + (tid >> 3) + 32 * i, row_end - 1);  // rows past the end repeat the last one
    xsrc[i] = (rows ? rows[gr] : gr) * width;
  }
  const int dst = tf_at(tid >> 3, tid & 7);  // (32 rows further on: the same permutation)

  const int stages = (width + TF_K - 1) / TF_K, kspan = stages * TF_K;
  const int rot = (width & 255) == 0 ? static_cast<int>((static_cast<unsigned>(col_block) * 3u) % stages) * TF_K : 0;
  const bool ragged = (width & (TF_K - 1)) != 0;
  auto place = [&](int k0, bool& ok) {
    k0 = min(k0, kspan - TF_K);
    const int k = (k0 + rot < kspan ? k0 + rot : k0 + rot - kspan) + kc_mine;
    ok = k < width;
    return ok ? k : 0;
  };
  f32x4 wreg[3][2], xreg[3][NPX];
  auto fetch = [&](int k0, f32x4 (&wr)[2], f32x4 (&xr)[NPX]) {
    bool ok;
    const int k = place(k0, ok);
#pragma unroll
    for (int i = 0; i < 2; ++i) wr[i] = *reinterpret_cast<const f32x4*>(w_expert + wsrc[i] + k);
#pragma unroll
    for (int i = 0; i < NPX; ++i) xr[i] = *reinterpret_cast<const f32x4*>(a + xsrc[i] + k);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto stage = [&](int k0, int buf, const f32x4 (&wr)[2], const f32x4 (&xr)[NPX]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4*>(ws + buf * TF_TILE + dst + 32 * TF_K * i) = wr[i];
#pragma unroll
    for (int i = 0; i < NPX; ++i) *reinterpret_cast<f32x4*>(xs + buf * TF_TILE + dst + 32 * TF_K * i) = xr[i];
    if (ragged) {
      bool ok;
      place(k0, ok);
      if (!ok) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4*>(ws + buf * TF_TILE + dst + 32 * TF_K * i) = zero;
#pragma unroll
        for (int i = 0; i < NPX; ++i) *reinterpret_cast<f32x4*>(xs + buf * TF_TILE + dst + 32 * TF_K * i) = zero;
      }
    }
  };
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int wat[2], xat[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    wat[h] = tf_at(16 * wave + m, 4 * h + g);
    xat[h] = tf_at(m, 4 * h + g);
  }
  auto multiply = [&](int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 wa = *reinterpret_cast<const f32x4*>(ws + buf * TF_TILE + wat[h]);
      f32x4 xb[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) xb[t] = *reinterpret_cast<const f32x4*>(xs + buf * TF_TILE + xat[h] + 16 * TF_K * t);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[j], xb[t][j], acc[t], 0, 0, 0);
    }
  };

  fetch(0, wreg[0], xreg[0]);
  fetch(TF_K, wreg[1], xreg[1]);
  fetch(2 * TF_K, wreg[2], xreg[2]);
  stage(0, 0, wreg[0], xreg[0]);
  fetch(3 * TF_K, wreg[0], xreg[0]);
  __syncthreads();
  // stage s lies in LDS buffer s & 1; register set (s + 1) % 3 holds the next one and then takes stage s + 4
#define TF_STAGE(K0, BUF, SET)                                    \
  {                                                               \
    stage((K0) + TF_K, 1 - (BUF), wreg[SET], xreg[SET]);          \
    fetch((K0) + 4 * TF_K, wreg[SET], xreg[SET]);                 \
    if ((K0) < kspan) multiply(BUF);                              \
    __builtin_amdgcn_sched_barrier(0);                            \
    __syncthreads();                                              \
  }
  for (int k0 = 0; k0 < kspan; k0 += 6 * TF_K) {  // whole turns only, as in moe_tiled.hip
    TF_STAGE(k0, 0, 1)
    TF_STAGE(k0 + TF_K, 1, 2)
    TF_STAGE(k0 + 2 * TF_K, 0, 0)
    TF_STAGE(k0 + 3 * TF_K, 1, 1)
    TF_STAGE(k0 + 4 * TF_K, 0, 2)
    TF_STAGE(k0 + 5 * TF_K, 1, 0)
  }
#undef TF_STAGE

  // lane holds the wavefront's weight rows 4 g + i of tile row 16 t + m; for gate|up lanes of g 0, 1 the gate's sums,
  // those of g 2, 3 (32 lanes on) the same columns' up sums
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int r = row0 + 16 * t + m;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = acc[t][i];
      if constexpr (GATE_UP) v[i] = ix_glu(v[i], __shfl_xor(v[i], 32, 64), glu_limit);
      else if (act) v[i] = v[i] > 0.f ? v[i] * v[i] : 0.f;  // the square of relu
    }
    if (r >= row_end || (GATE_UP && g >= 2)) continue;
    const int nb = n0 + (GATE_UP ? 8 : 16) * wave + 4 * g;
    float* o = out + static_cast<int64_t>(r) * n_out + nb;
    if (nb + 4 <= n_out && (n_out & 3) == 0) {
      *reinterpret_cast<f32x4*>(o) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (nb + i < n_out) o[i] = v[i];
    }
  }
}

template <bool GATE_UP>
__global__ void __launch_bounds__(256, 4)
moe_grouped_tiled_f32_kernel(const float* a, const float* w, float* out, const int32_t* __restrict__ offsets,
                             const int32_t* __restrict__ rows, const int32_t* __restrict__ tile_expert,
                             const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_info, int n_out,
                             int width, int n_col_blocks, int act, float glu_limit) {
  __shared__ __attribute__((aligned(16))) float ws[2 * TF_TILE];
  __shared__ __attribute__((aligned(16))) float xs[2 * TF_TILE];
  // Workgroups go to the chip's eight dies in turn.  The (row tile, column block) pairs, tile by tile, are cut into eight
  // equal runs, one a die: the column blocks of a tile, which read the same activations, share an L2, and no die has more
  // of them than another (whole tiles dealt to the dies in turn: of 60, four dies had eight and four seven).
  const unsigned n_pairs = static_cast<unsigned>(tile_info[0]) * n_col_blocks, die = blockIdx.x & 7;
  auto cut = [&](unsigned d) { return static_cast<unsigned>(static_cast<uint64_t>(n_pairs) * d >> 3); };
  const unsigned pair = cut(die) + (blockIdx.x >> 3);
  if (pair >= cut(die + 1)) return;
  const int tile = static_cast<int>(pair / n_col_blocks), col_block = static_cast<int>(pair % n_col_blocks);
  const int e = tile_expert[tile], row0 = tile_row0[tile], row_end = offsets[e + 1];
  const int held = min(TF_ROWS, row_end - row0);
  if (held <= 0) return;
#define BODY(NT) \
  tiled_f32_body<GATE_UP, NT>(a, w, out, rows, n_out, width, e, row0, row_end, col_block, ws, xs, act, glu_limit)
  switch ((held + 15) >> 4) {
    case 1: BODY(1); break;
    case 2: BODY(2); break;
    case 3: BODY(3); break;
    default: BODY(4); break;
  }
#undef BODY
}

// Shapes as ix_moe_grouped_plain, all float32; the row-tile map must have been made for tiles of 64 rows; operands on
// 16-byte boundaries.  gate_up: 0 a plain product, 1 gate|up rows with SwiGLU (glu_limit: see `ix_glu`), 2 a plain
// product whose results pass the square of relu.
extern "C" int ix_moe_grouped_tiled_f32(const float* a, const float* w, float* out, const int32_t* offsets,
                                        const int32_t* rows, const int32_t* tile_expert, const int32_t* tile_row0,
                                        const int32_t* tile_info, int max_tiles, int64_t a_rows, int64_t n_out,
                                        int64_t width, int gate_up, float glu_limit, hipStream_t stream) {
  IX_REQUIRE(n_out > 0 && width > 0 && max_tiles >= 0, "sizes must be positive");
  IX_REQUIRE(width % 4 == 0, "the reduction width must be a multiple of 4");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) & 15) == 0,
             "operands must lie on 16-byte boundaries");
  IX_REQUIRE(n_out < (1 << 30) && width < (1 << 30), "sizes too large");
  IX_REQUIRE(a_rows >= 0 && a_rows * width < (int64_t(1) << 31) && (gate_up == 1 ? 2 : 1) * n_out * width < (int64_t(1) << 31),
             "the activations, and one expert's weights, must hold fewer than 2^31 numbers");
  IX_REQUIRE(gate_up >= 0 && gate_up <= 2, "gate_up must be 0, 1 or 2");
  IX_REQUIRE(max_tiles <= 65535, "too many row tiles for one launch");
  if (max_tiles == 0) return 0;
  const int cols = gate_up == 1 ? TF_WROWS / 2 : TF_WROWS;
  const int n_col_blocks = static_cast<int>((n_out + cols - 1) / cols);
  const int64_t groups = 8 * (static_cast<int64_t>(n_col_blocks) * max_tiles / 8 + 2);  // (a die has at most this many pairs)
  IX_REQUIRE(groups < (int64_t(1) << 31), "too many workgroups for one launch");
  dim3 grid(static_cast<unsigned>(groups)), block(256);
  if (gate_up == 1)
    hipLaunchKernelGGL((moe_grouped_tiled_f32_kernel<true>), grid, block, 0, stream, a, w, out, offsets, rows, tile_expert,
                       tile_row0, tile_info, (int)n_out, (int)width, n_col_blocks, 0, glu_limit);
  else
    hipLaunchKernelGGL((moe_grouped_tiled_f32_kernel<false>), grid, block, 0, stream, a, w, out, offsets, rows, tile_expert,
                       tile_row0, tile_info, (int)n_out, (int)width, n_col_blocks, gate_up == 2 ? 1 : 0, glu_limit);
  return ix_check_launch("ix_moe_grouped_tiled_f32");
}
