// Grouped expert products in float32 for more than a few rows per expert (prompt portions of a float32 run): operands
// staged through LDS, v_mfma_f32_16x16x4_f32, every product and sum in 32 bits.
//
// What bounds it: at a few dozen rows per expert the weights' way from memory, from about fifty on the matrix cores
// (32 cycles for 16 x 16 x 4).  A workgroup owns up to 64 rows of one expert (a tile of the grouping kernel's map: with
// a few hundred tokens all rows of an expert, so that its weights come from memory once) x one or two blocks of 64 weight rows, which for
// gate|up are 32 gate rows and their 32 up rows; its four wavefronts take sixteen weight rows of each (for gate|up of one block
// eight and eight, of two sixteen and sixteen) and all of the tile's rows.  Stages of 32 of the reduction (128 bytes a row) go through a
// ring of three to six LDS buffers that the loads fill by themselves, with one barrier a stage, as in moe_tiled.hip; half a
// compute unit's LDS, so that two workgroups share one and one's products overlap with the other's waits.  Rows of LDS keep
// their eight 16-byte pieces permuted (piece p of row r at p ^ ((r >> 1) & 7)), so that sixteen rows read at one piece fall on
// different banks.  The weights of an expert with one tile go past the caches if their rows are whole lines (42 experts of 2,048 on 2,308, 193
// tokens of two, gate|up 333 us past them, 269 through them, as rows and stages share lines).
//
// A lane reads four consecutive numbers of its row at a time; product j of a piece multiplies the j-th of them, so the
// four slots of the reduction that one matrix instruction adds up are the pieces' j-th numbers, the same in both
// operands.  Blocks of weight rows start the reduction at a stage that follows from their number and wrap round: rows of a
// power of two bytes would otherwise all ask the same memory channels at once.  The order of a result's sum so depends
// on its column alone (two scores of a later router that are 1e-6 apart fall the other way with another order).
//
// Two blocks read a tile's activations for half as many workgroups; one block has twice the workgroups, each with half the
// products.  Which of them, by the workgroups that two would give, the sizes' geometric mean of one product's time (509 shapes of 4 to
// 128 experts, widths of 512 to 2,560, 40 to 1,024 tokens), two blocks against one: up to 128 1.78, 256 1.38, 512 1.21, 768
// 1.08, 1,024 1.06, 1,500 1.03, more 0.99 (8 experts of 768 on 2,048, 128 tokens, both products: 116 us, 68 with one).
// With reductions of 256, 512 and 768 the three stages more that two turned blocks walk weigh too much, so they stay with one (128
// experts of 256, down to 2,560, 74 tokens of six, 57 us with two blocks, 49 with one; eight of 512 on 512, 1,105 tokens 125 and 109).
//
// Measured with 60 experts of 1,408 on a width of 2,048, 4 a token, unevenly routed, both products, us, two blocks against pieces through
// registers and LDS writes, one block, a die's run of tiles in their order: 170 tokens 389 -> 348, 361 503 -> 415, 511 562
// -> 490, 800 747 -> 648; 32 rows each 428 -> 404, 64 rows each 662 -> 641 (the weights alone take 324, the last one's products
// 474).  Of it at 511 tokens the direct loads and 128 rows 50 to 65, the order of the tiles 45 to 60; that both blocks of a
// workgroup keep their own order of sums costs 30.
#include <type_traits>

#include "lds_loads.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define TF_ROWS 64     // rows of a tile of the map
#define TF_K 32        // numbers of the reduction per stage
#define TF_APART 3     // stages between the starts of neighbouring blocks of 64 weight rows
#define TF_TURNED_WIDTH 1024
#define TF_LDS 81920   // bytes: half a compute unit's
__device__ __forceinline__ int tf_at(int row, int piece) { return row * TF_K + ((piece ^ ((row >> 1) & 7)) << 2); }

// BLOCKS: blocks of 64 weight rows that the workgroup owns, one or two.  NT: sixteens of rows that the tile holds.  Every load
// is unconditional: a stage past the end asks for the last stage again, a piece past the row's end for the row's last one, with
// zeros in its place among the operands.
template <bool GATE_UP, int NT, bool ONCE, int BLOCKS>
__device__ __forceinline__ void tiled_f32_body(const float* a, const float* w, float* out,
                                               const int32_t* __restrict__ rows, int n_out, int width, int e, int row0,
                                               int row_end, int col_block, float* lds, int act, float glu_limit) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  constexpr int COLS = (GATE_UP ? 32 : 64) * BLOCKS;
  constexpr int NPW = 2 * BLOCKS, NPX = (NT + 1) / 2;  // loads of a wavefront a stage, eight rows each
  constexpr int RING = BLOCKS == 2 ? (NT <= 2 ? 4 : 3) : (NT <= 2 ? 6 : 5);  // stages that LDS holds
  constexpr unsigned WT = 64 * BLOCKS * 4 * TF_K, XT = 32 * NPX * 4 * TF_K;  // bytes of a stage
  static_assert(RING * (WT + XT) <= TF_LDS, "the rings fit");
  const int n0 = col_block * COLS;

  const int64_t w_rows = GATE_UP ? 2 * static_cast<int64_t>(n_out) : n_out;
  const float* w_expert = w + static_cast<int64_t>(e) * w_rows * width;
  int64_t wsrc[NPW], xsrc[NPX];  // where this lane's rows start, in numbers
#pragma unroll
  for (int i = 0; i < NPW; ++i) {
    // LDS row; wavefront r / (16 BLOCKS) multiplies it, for gate|up 8 BLOCKS gate rows, then their up rows
    const int r = 8 * (wave + 4 * i) + (lane >> 3), of = r / (16 * BLOCKS), in = r % (8 * BLOCKS);
    const int src = GATE_UP ? ((r & (8 * BLOCKS)) ? n_out : 0) + min(n0 + 8 * BLOCKS * of + in, n_out - 1) : min(n0 + r, n_out - 1);
    wsrc[i] = static_cast<int64_t>(src) * width;
  }
#pragma unroll
  for (int i = 0; i < NPX; ++i) {
    const int gr = min(row0 + 8 * (wave + 4 * i) + (lane >> 3), row_end - 1);  // rows past the end repeat the last one
    xsrc[i] = static_cast<int64_t>(rows ? rows[gr] : gr) * width;
  }
  const int piece = 4 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4)));  // what belongs at piece lane & 7 of the lane's rows

  // Blocks of 64 weight rows start the reduction at a stage that follows from their number and wrap round.  The two of a
  // workgroup that owns two start TF_APART stages apart: it walks so many stages more, the first of them for the first two
  // wavefronts only and the last of them for the others (and asks for all rows in each, so for 3 stages of every row twice).
  const int stages = (width + TF_K - 1) / TF_K;
  const bool turned = (width & 255) == 0;  // (then there are eight stages at least)
  const int total = stages + (BLOCKS == 2 && turned ? TF_APART : 0);
  const int begin = turned ? static_cast<int>((static_cast<unsigned>(col_block) * (unsigned{BLOCKS} * TF_APART)) % stages) : 0;
  auto place = [&](int s) {  // where stage s starts in a row (past the end: the last stage again)
    int k = min(s, total - 1) + begin;
    k = k < stages ? k : k - stages;
    return (k < stages ? k : k - stages) * TF_K;
  };
  auto mine = [&](int s) { return BLOCKS == 1 || !turned || (wave < 2 ? s < stages : s >= TF_APART); };
  auto load = [&](int buf, int i, int at) {  // the i-th of a stage's loads
    if (i < NPX) lds_load16<false>(lds, RING * WT + buf * XT + 1024 * (wave + 4 * i), a + xsrc[i] + at);
    else if (i < NPX + NPW) lds_load16<ONCE>(lds, buf * WT + 1024 * (wave + 4 * (i - NPX)), w_expert + wsrc[i - NPX] + at);
  };
  auto at_stage = [&](int s) { return min(place(s) + piece, width - 4); };

  f32x4 acc[BLOCKS][NT];
#pragma unroll
  for (int b = 0; b < BLOCKS; ++b)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int at16[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) at16[h] = tf_at(m, 4 * h + g);
  const float* const ws = lds + 16 * BLOCKS * wave * TF_K;
  const float* const xs = lds + RING * WT / 4;
  struct Half { f32x4 w[BLOCKS], x[NT]; };
  Half h0, h1;
  auto read = [&](Half& h, int i, int buf, int half) {  // the i-th of a half's NT + BLOCKS pieces
    if (i < BLOCKS) h.w[i] = *reinterpret_cast<const f32x4*>(ws + buf * (WT / 4) + at16[half] + 16 * i * TF_K);
    else if (i < NT + BLOCKS) h.x[i - BLOCKS] = *reinterpret_cast<const f32x4*>(xs + buf * (XT / 4) + at16[half] + 16 * (i - BLOCKS) * TF_K);
  };
  auto products = [&](const Half& h, int j) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b) acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(h.w[b][j], h.x[t][j], acc[b][t], 0, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < RING; ++s)
#pragma unroll
    for (int i = 0; i < NPX + NPW; ++i) load(s, i, at_stage(s));
  wait_loads<(NPX + NPW) * (RING - 1)>();
  lds_barrier();
  int buf = 0;
#pragma unroll
  for (int i = 0; i < NT + BLOCKS; ++i) read(h0, i, buf, 0);
  constexpr int READS = (NT + BLOCKS + 1) / 2, LOADS = (NPX + NPW + 2) / 3;
  auto stage = [&](auto left, int s) {
    constexpr int LEFT = decltype(left)::value;  // at least so many stages follow
    if constexpr (LEFT == 0) {
#pragma unroll
      for (int i = 0; i < NT + BLOCKS; ++i) read(h1, i, buf, 1);
      if (width & (TF_K - 1)) {  // the last stage is not whole
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int half = 0; half < 2; ++half)
          if (place(s) + 16 * half + 4 * g >= width) {
            Half& h = half ? h1 : h0;
#pragma unroll
            for (int b = 0; b < BLOCKS; ++b) h.w[b] = zero;
#pragma unroll
            for (int t = 0; t < NT; ++t) h.x[t] = zero;
          }
      }
      if (mine(s)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) products(h0, j);
#pragma unroll
        for (int j = 0; j < 4; ++j) products(h1, j);
      }
    } else {
      const bool own = mine(s);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (own) products(h0, j);
#pragma unroll
        for (int i = READS * j; i < READS * (j + 1); ++i) read(h1, i, buf, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      wait_loads<(NPX + NPW) * (RING - 2 < LEFT - 1 ? RING - 2 : LEFT - 1)>();  // stage s + 1 has landed
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
      const int free = buf;  // nobody reads stage s any more
      buf = buf + 1 == RING ? 0 : buf + 1;
      const int at = LEFT >= RING ? at_stage(s + RING) : 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (own) products(h1, j);
#pragma unroll
        for (int i = READS * j; i < READS * (j + 1); ++i) read(h0, i, buf, 0);
        if constexpr (LEFT >= RING)
#pragma unroll
          for (int i = LOADS * j; i < LOADS * (j + 1); ++i) load(free, i, at);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
#define TF_STAGE(LEFT, S) stage(std::integral_constant<int, (LEFT)>{}, (S))
  for (int s = 0; s < total - RING; ++s) TF_STAGE(RING, s);
  if constexpr (RING > 5)
    if (total > 5) TF_STAGE(5, total - 6);
  if constexpr (RING > 4)
    if (total > 4) TF_STAGE(4, total - 5);
  if constexpr (RING > 3)
    if (total > 3) TF_STAGE(3, total - 4);
  if (total > 2) TF_STAGE(2, total - 3);
  if (total > 1) TF_STAGE(1, total - 2);
  TF_STAGE(0, total - 1);
#undef TF_STAGE
  wait_loads<0>();  // (with fewer stages than the ring holds, the last one again)

  // lane holds weight rows (sixteen) + 4 g + i of tile row 16 t + m; for gate|up of one block lanes of g 0, 1 the gate's sums,
  // those of g 2, 3 (32 lanes on) the same columns' up sums
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int r = row0 + 16 * t + m;
#pragma unroll
    for (int b = 0; b < (GATE_UP ? 1 : BLOCKS); ++b) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = acc[b][t][i];
        if constexpr (GATE_UP) v[i] = ix_glu(v[i], BLOCKS == 2 ? acc[BLOCKS - 1][t][i] : __shfl_xor(v[i], 32, IX_WAVE), glu_limit);
        else if (act) v[i] = v[i] > 0.f ? v[i] * v[i] : 0.f;  // the square of relu
      }
      if (r >= row_end || (GATE_UP && BLOCKS == 1 && g >= 2)) continue;
      const int nb = n0 + (GATE_UP ? 8 : 16) * BLOCKS * wave + 16 * b + 4 * g;
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
}

template <bool GATE_UP, int BLOCKS>
__global__ void __launch_bounds__(256, 2)
moe_grouped_tiled_f32_kernel(const float* a, const float* w, float* out, const int32_t* __restrict__ offsets,
                             const int32_t* __restrict__ rows, const int32_t* __restrict__ tile_expert,
                             const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_info, int n_out,
                             int width, int n_col_blocks, int act, float glu_limit) {
  __shared__ __attribute__((aligned(1024))) float lds[TF_LDS / 4];
  // The tiles with most rows come first, so that what is left at the end is short, and a tile's column blocks go to the
  // chip's eight dies in turn, so that each has as much of it (a die's run of whole tiles took 133 to 178 us at 511 tokens).  Tiles of as
  // many sixteens stay together in the map's order; beyond 512 of them the end no longer matters.  (Long and short tiles in
  // turn leave half the chip idle at times: workgroups are handed out in order, each to a place of its own.)
  const int n_tiles = tile_info[0];
  const unsigned pair = blockIdx.x;
  if (pair >= static_cast<unsigned>(n_tiles) * n_col_blocks) return;
  int tile = static_cast<int>(pair / n_col_blocks);
  const int col_block = static_cast<int>(pair % n_col_blocks);
  if (n_tiles <= 8 * 64) {
    const int lane = threadIdx.x & 63;
    unsigned sixteens = 0;  // of the tile 64 c + lane, in four bits for each c
    int count[5] = {0, 0, 0, 0, 0};
    for (int c = 0; 64 * c < n_tiles; ++c) {
      const int t = 64 * c + lane;
      int n = 0;
      if (t < n_tiles) n = max(1, (min(TF_ROWS, offsets[tile_expert[t] + 1] - tile_row0[t]) + 15) >> 4);
      sixteens |= static_cast<unsigned>(n) << (4 * c);
#pragma unroll
      for (int k = 1; k <= 4; ++k) count[k] += __popcll(__ballot(n == k));
    }
    int place = tile, kind = 4;  // the place among the tiles of so many sixteens
#pragma unroll
    for (int k = 4; k > 1; --k)
      if (kind == k && place >= count[k]) {
        place -= count[k];
        kind = k - 1;
      }
    for (int c = 0; 64 * c < n_tiles; ++c) {
      unsigned long long of_kind = __ballot(static_cast<int>(sixteens >> (4 * c) & 15) == kind);
      const int n = __popcll(of_kind);
      if (place < n) {
        for (; place > 0; --place) of_kind &= of_kind - 1;
        tile = 64 * c + __ffsll(of_kind) - 1;
        break;
      }
      place -= n;
    }
    tile = __builtin_amdgcn_readfirstlane(tile);
  }
  const int e = tile_expert[tile], row0 = tile_row0[tile], row_end = offsets[e + 1];
  const int held = min(TF_ROWS, row_end - row0);
  if (held <= 0) return;
  // an expert's only tile: its weights are read once, past the caches, if its rows are whole lines
  const bool once = held == row_end - offsets[e] && ((width & 31) | static_cast<int>(reinterpret_cast<uintptr_t>(w) & 127)) == 0;
#define CALL(NT, ONCE) \
  tiled_f32_body<GATE_UP, NT, ONCE, BLOCKS>(a, w, out, rows, n_out, width, e, row0, row_end, col_block, lds, act, glu_limit)
#define BODY(NT) if (once) CALL(NT, true); else CALL(NT, false)
  switch ((held + 15) >> 4) {
    case 1: BODY(1); break;
    case 2: BODY(2); break;
    case 3: BODY(3); break;
    default: BODY(4); break;
  }
#undef BODY
#undef CALL
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
  const auto column_blocks = [&](int blocks) {
    const int cols = (gate_up == 1 ? 32 : 64) * blocks;
    return (n_out + cols - 1) / cols;
  };
  // (see the top of the file; with short reductions the three stages more that two turned blocks walk weigh too much)
  const int blocks = column_blocks(2) * max_tiles <= 1024 || (width % 256 == 0 && width < TF_TURNED_WIDTH) ? 1 : 2;
  const int n_col_blocks = static_cast<int>(column_blocks(blocks));
  const int64_t groups = static_cast<int64_t>(n_col_blocks) * max_tiles;
  IX_REQUIRE(groups < (int64_t(1) << 31), "too many workgroups for one launch");
  dim3 grid(static_cast<unsigned>(groups)), block(256);
#define LAUNCH(GU, BLOCKS)                                                                                                  \
  hipLaunchKernelGGL((moe_grouped_tiled_f32_kernel<GU, BLOCKS>), grid, block, 0, stream, a, w, out, offsets, rows,          \
                     tile_expert, tile_row0, tile_info, (int)n_out, (int)width, n_col_blocks, gate_up == 2 ? 1 : 0, glu_limit)
  if (gate_up == 1) {
    if (blocks == 2) LAUNCH(true, 2);
    else LAUNCH(true, 1);
  } else {
    if (blocks == 2) LAUNCH(false, 2);
    else LAUNCH(false, 1);
  }
#undef LAUNCH
  return ix_check_launch("ix_moe_grouped_tiled_f32");
}
