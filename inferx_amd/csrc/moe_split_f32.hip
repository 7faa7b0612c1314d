// Grouped expert products in float32 for more than a few rows per expert (prompt portions of a float32 run), on the bfloat16
// matrix cores (see split_f32.h): what moe_tiled_f32.hip does with the float32 instructions, where rows are whole stages of 32.
//
// What bounds it: the weights' way from memory.  60 experts of 1,408 on a width of 2,048, four a token, unevenly routed, both products, us,
// the float32 instructions / here (the weights alone 216 + 108): 150 tokens 194 + 102 / 190 + 101, 256 240 + 119 / 206 + 117, 400 288 + 139 /
// 240 + 120, 511 332 + 166 / 281 + 140, 700 428 + 208 / 345 + 177.  (Eight wavefronts with 256 weight rows and all of a compute unit's LDS:
// 290 + 149 at 511.)
//
// A workgroup of four wavefronts owns up to 64 rows of one expert (a tile of the grouping kernel's map) x 128 weight rows, for gate|up 64 gate
// rows and their up rows; a wavefront 32 of them (for gate|up sixteen and sixteen, so that it holds both sums of a column), which it
// alone splits, x all of the tile's rows in one or two blocks of 32.  The activations are split beforehand
// (`ix_split_rows`).  Stages of 32 of the reduction go through rings of LDS buffers that the loads fill by themselves, half a
// compute unit's LDS, so that two workgroups share one.  The order of a result's sum depends on its column alone.
#include <type_traits>

#include "lds_loads.h"
#include "moe_tiled_f32.h"
#include "split_f32.h"

#define MS_K 32      // numbers of the reduction a stage
#define MS_ROW 192   // bytes of an activation row's stage: 64 of each part
#define MS_W 128     // weight rows of a workgroup
#define MS_LDS 81920  // bytes: half a compute unit's
// piece p (of eight) of weight row r lies at p ^ ((r >> 1) & 7); piece p (of twelve, four a part) of activation row r at p ^ ((r >> 2) & 3)
__device__ __forceinline__ int ms_weight_at(int row, int piece) { return row * 4 * MS_K + ((piece ^ ((row >> 1) & 7)) << 4); }
__device__ __forceinline__ int ms_row_at(int row, int piece) { return row * MS_ROW + ((piece ^ ((row >> 2) & 3)) << 4); }

// XB: blocks of 32 rows that the tile holds.
template <bool GATE_UP, int XB, bool ONCE>
__device__ __forceinline__ void split_body(const float* a, const __bf16* parts, const float* w, float* out, const int32_t* __restrict__ rows,
                                           int n_out, int width, int e, int row0, int row_end, int col_block, char* lds, int act,
                                           float glu_limit) {
  constexpr int RING_W = 3, RING_X = XB == 1 ? 3 : 2;  // stages that LDS holds
  constexpr unsigned WT = MS_W * 4 * MS_K, XT = XB == 1 ? 8192 : 12288;  // bytes of a stage (one block of rows: and 2 KB that nobody reads)
  constexpr int NPW = WT / 4096, NPX = XT / 4096;                        // loads of a wavefront a stage
  static_assert(RING_W * WT + RING_X * XT <= MS_LDS, "the rings fit");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 31, g = lane >> 5;
  const int n0 = col_block * (GATE_UP ? MS_W / 2 : MS_W);

  const float* const w_expert = w + static_cast<int64_t>(e) * (GATE_UP ? 2 * static_cast<int64_t>(n_out) : n_out) * width;
  // where this lane's pieces of a stage start, in bytes
  int64_t wsrc[NPW], xsrc[NPX];
#pragma unroll
  for (int i = 0; i < NPW; ++i) {
    const int r = 8 * (wave + 4 * i) + (lane >> 3), p = (lane & 7) ^ ((r >> 1) & 7);
    const int row = GATE_UP ? ((r & 16) ? n_out : 0) + min(n0 + 16 * (r / 32) + (r & 15), n_out - 1) : min(n0 + r, n_out - 1);
    wsrc[i] = 4 * (static_cast<int64_t>(row) * width) + 16 * p;
  }
#pragma unroll
  for (int i = 0; i < NPX; ++i) {
    const int at = 64 * (wave + 4 * i) + lane, r = at / 12, p = (at % 12) ^ ((r >> 2) & 3);
    const int gr = min(row0 + r, row_end - 1);  // rows past the end repeat the last one
    xsrc[i] = 6 * (static_cast<int64_t>(rows ? rows[gr] : gr) * width) + 16 * p;
  }
  // (blocks of weight rows start the reduction at different stages and wrap round, see moe_tiled_f32.hip)
  const int stages = width / MS_K;
  const int rot = width % 256 == 0 ? static_cast<int>((static_cast<unsigned>(col_block) * 3u) % static_cast<unsigned>(stages)) : 0;
  auto place = [&](int s) {  // (past the end: the last stage again)
    const int k = min(s, stages - 1) + rot;
    return k < stages ? k : k - stages;
  };
  auto load_w = [&](unsigned buf, int i, int stage) {
    lds_load16<ONCE>(lds, buf + 1024 * (wave + 4 * i), reinterpret_cast<const char*>(w_expert) + wsrc[i] + 4 * MS_K * stage);
  };
  auto load_x = [&](unsigned buf, int i, int stage) {
    lds_load16<false>(lds, RING_W * WT + buf + 1024 * (wave + 4 * i), reinterpret_cast<const char*>(parts) + xsrc[i] + MS_ROW * stage);
  };

  f32x16 large[XB], small[XB];
#pragma unroll
  for (int t = 0; t < XB; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) large[t][i] = small[t][i] = 0.f;
  int w_at[2][2], x_at[2][3];  // half of the stage; piece of the lane's two, part
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
    for (int p = 0; p < 2; ++p) w_at[kk][p] = ms_weight_at(m, 4 * kk + 2 * g + p);
#pragma unroll
    for (int p = 0; p < 3; ++p) x_at[kk][p] = ms_row_at(m, 4 * p + 2 * kk + g);
  }
  const char* const ws = lds + 32 * wave * 4 * MS_K;
  const char* const xs = lds + RING_W * WT;
  struct Half { bf16x8 w[3], x[XB][3]; };
  Half h0, h1;
  f32x4 raw[2];
  auto read = [&](Half& h, unsigned wbuf, unsigned xbuf, int kk) {  // the weights as they are, the activations' parts
#pragma unroll
    for (int p = 0; p < 2; ++p) raw[p] = *reinterpret_cast<const f32x4*>(ws + wbuf + w_at[kk][p]);
#pragma unroll
    for (int t = 0; t < XB; ++t)
#pragma unroll
      for (int p = 0; p < 3; ++p) h.x[t][p] = *reinterpret_cast<const bf16x8*>(xs + xbuf + 32 * t * MS_ROW + x_at[kk][p]);
  };
  auto products = [&](const Half& h) {
    auto add = [&](f32x16 (&sum)[XB], int p, int q) {
#pragma unroll
      for (int t = 0; t < XB; ++t) sum[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h.w[p], h.x[t][q], sum[t], 0, 0, 0);
    };
    add(small, 0, 2);
    add(large, 0, 0);
    add(small, 2, 0);
    add(small, 1, 1);
    add(small, 0, 1);
    add(small, 1, 0);
  };
  // a half's products with the next one's splitting between them
  auto interleave = [&]() {
#pragma unroll
    for (int i = 0; i < 6 * XB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x2, 8 / XB, 0);
    }
  };

#pragma unroll
  for (int s = 0; s < RING_W; ++s) {
    const int at = place(s);
    if (s < RING_X)
#pragma unroll
      for (int i = 0; i < NPX; ++i) load_x(s * XT, i, at);
#pragma unroll
    for (int i = 0; i < NPW; ++i) load_w(s * WT, i, at);
  }
  wait_loads<NPW * (RING_W - 1) + NPX * (RING_X - 1)>();
  lds_barrier();
  unsigned wbuf = 0, xbuf = 0;
  read(h0, 0, 0, 0);
  split8(raw[0], raw[1], h0.w);
  read(h1, 0, 0, 1);
  // Stage s, the first half's operands ready, the second half's on their way from LDS; LEFT: at least so many stages follow.
  auto stage = [&](auto left, int s) {
    constexpr int LEFT = decltype(left)::value;
    __builtin_amdgcn_sched_barrier(0);
    products(h0);
    split8(raw[0], raw[1], h1.w);
    interleave();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (LEFT > 0) {
      // Stage s + 1 must have landed; after its last load there were issued (an iteration issues activations first) those of the
      // stages after it that the rings hold, as far as there are so many.
      constexpr int LATER_W = RING_W - 2 < LEFT - 1 ? RING_W - 2 : LEFT - 1, LATER_X = RING_X - 2 < LEFT - 1 ? RING_X - 2 : LEFT - 1;
      wait_loads<NPW * LATER_W + NPX * LATER_X>();
      lds_barrier();
      const unsigned wfree = wbuf, xfree = xbuf;  // nobody reads stage s any more
      wbuf = wbuf + WT == RING_W * WT ? 0 : wbuf + WT;
      xbuf = xbuf + XT == RING_X * XT ? 0 : xbuf + XT;
      read(h0, wbuf, xbuf, 0);
      if constexpr (LEFT >= RING_X) {
        const int at = place(s + RING_X);
#pragma unroll
        for (int i = 0; i < NPX; ++i) load_x(xfree, i, at);
      }
      if constexpr (LEFT >= RING_W) {
        const int at = place(s + RING_W);
#pragma unroll
        for (int i = 0; i < NPW; ++i) load_w(wfree, i, at);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    products(h1);
    if constexpr (LEFT > 0) {
      split8(raw[0], raw[1], h0.w);
      interleave();
      __builtin_amdgcn_sched_barrier(0);
      read(h1, wbuf, xbuf, 1);
    }
  };
  for (int s = 0; s < stages - RING_W; ++s) stage(std::integral_constant<int, RING_W>{}, s);
  if (stages > 2) stage(std::integral_constant<int, 2>{}, stages - 3);
  if (stages > 1) stage(std::integral_constant<int, 1>{}, stages - 2);
  stage(std::integral_constant<int, 0>{}, stages - 1);
  wait_loads<0>();  // (with fewer stages than the rings hold, the last one again)

  // lane holds rows 32 wave + 8 q + 4 g + i of the weight rows and tile row 32 t + m; for gate|up q 0, 1 are gate rows, q 2, 3 their up rows
#pragma unroll
  for (int t = 0; t < XB; ++t) {
    const int r = row0 + 32 * t + m;
    if (r >= row_end) continue;
    auto sum = [&](int q, int i) { return large[t][4 * q + i] + small[t][4 * q + i]; };
#pragma unroll
    for (int q = 0; q < (GATE_UP ? 2 : 4); ++q) {
      const int nb = n0 + (GATE_UP ? 16 : 32) * wave + 8 * q + 4 * g;
      float v[4], u[4];
      bool numbers = true;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = sum(q, i);
        u[i] = GATE_UP ? sum(q + 2 * GATE_UP, i) : 0.f;
        numbers = numbers && is_number(v[i]) && is_number(u[i]);
      }
      if (!numbers) {
        const float* const row = a + static_cast<int64_t>(rows ? rows[r] : r) * width;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nb + i < n_out) {
            v[i] = plain_dot(row, w_expert + static_cast<int64_t>(nb + i) * width, width);
            if (GATE_UP) u[i] = plain_dot(row, w_expert + static_cast<int64_t>(n_out + nb + i) * width, width);
          }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (GATE_UP) v[i] = ix_glu(v[i], u[i], glu_limit);
        else if (act) v[i] = v[i] > 0.f ? v[i] * v[i] : 0.f;  // the square of relu
      }
      float* const o = out + static_cast<int64_t>(r) * n_out + nb;
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

template <bool GATE_UP>
__global__ void __launch_bounds__(256, 2)
moe_grouped_split_kernel(const float* a, const __bf16* parts, const float* w, float* out, const int32_t* __restrict__ offsets,
                         const int32_t* __restrict__ rows, const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_row0,
                         const int32_t* __restrict__ tile_info, int n_out, int width, int n_col_blocks, int act, float glu_limit) {
  __shared__ __attribute__((aligned(1024))) char lds[MS_LDS];
  const int n_tiles = tile_info[0];
  const unsigned pair = blockIdx.x;
  if (pair >= static_cast<unsigned>(n_tiles) * n_col_blocks) return;
  const int tile = tf_tile(static_cast<int>(pair / n_col_blocks), n_tiles, offsets, tile_expert, tile_row0);
  const int col_block = static_cast<int>(pair % n_col_blocks);
  const int e = tile_expert[tile], row0 = tile_row0[tile], row_end = min(offsets[e + 1], row0 + TF_ROWS), held = row_end - row0;
  if (held <= 0) return;
  // an expert's only tile: its weights are read once, past the caches (their rows are whole lines)
  const bool once = held == offsets[e + 1] - offsets[e] && (reinterpret_cast<uintptr_t>(w) & 127) == 0;
#define CALL(XB, ONCE) \
  split_body<GATE_UP, XB, ONCE>(a, parts, w, out, rows, n_out, width, e, row0, row_end, col_block, lds, act, glu_limit)
  if (held <= 32) {
    if (once) CALL(1, true);
    else CALL(1, false);
  } else {
    if (once) CALL(2, true);
    else CALL(2, false);
  }
#undef CALL
}

// As ix_moe_grouped_tiled_f32, with a width in multiples of 32; parts: `ix_split_rows` of a.
extern "C" int ix_moe_grouped_split(const float* a, const void* parts, const float* w, float* out, const int32_t* offsets,
                                    const int32_t* rows, const int32_t* tile_expert, const int32_t* tile_row0,
                                    const int32_t* tile_info, int max_tiles, int64_t n_out, int64_t width, int gate_up,
                                    float glu_limit, hipStream_t stream) {
  IX_REQUIRE(n_out > 0 && width > 0 && max_tiles >= 0, "sizes must be positive");
  IX_REQUIRE(width % MS_K == 0, "the reduction width must be a multiple of 32");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(parts) | reinterpret_cast<uintptr_t>(w) |
               reinterpret_cast<uintptr_t>(out)) & 15) == 0,
             "operands must lie on 16-byte boundaries");
  IX_REQUIRE(n_out < (1 << 30) && width < (1 << 30), "sizes too large");
  IX_REQUIRE(gate_up >= 0 && gate_up <= 2, "gate_up must be 0, 1 or 2");
  IX_REQUIRE(max_tiles <= 65535, "too many row tiles for one launch");
  if (max_tiles == 0) return 0;
  const int cols = gate_up == 1 ? MS_W / 2 : MS_W, n_col_blocks = static_cast<int>((n_out + cols - 1) / cols);
  const int64_t groups = static_cast<int64_t>(n_col_blocks) * max_tiles;
  IX_REQUIRE(groups < (int64_t(1) << 31), "too many workgroups for one launch");
#define LAUNCH(GU)                                                                                                             \
  hipLaunchKernelGGL(moe_grouped_split_kernel<GU>, dim3(static_cast<unsigned>(groups)), dim3(256), 0, stream, a, (const __bf16*)parts, w, \
                     out, offsets, rows, tile_expert, tile_row0, tile_info, (int)n_out, (int)width, n_col_blocks, gate_up == 2 ? 1 : 0,  \
                     glu_limit)
  if (gate_up == 1) LAUNCH(true);
  else LAUNCH(false);
#undef LAUNCH
  return ix_check_launch("ix_moe_grouped_split");
}
