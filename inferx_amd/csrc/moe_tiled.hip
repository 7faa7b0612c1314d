// Grouped expert products for many rows per expert (prompt portions), bfloat16,
// staged through LDS.  Same results as moe_mfma.hip's kernel; that one streams
// each operand per wavefront, which is right when the weights are the traffic
// (decoding) and wasteful when dozens of rows share them.
//
// A workgroup owns up to 160 rows of one expert, 192 in the wide form (a row
// tile of the grouping kernel's map; with a few hundred tokens that is all rows
// of the expert, so its weights are read once) x 128 weight rows: for the gate|up product 64 gate
// rows and the 64 up rows that belong to them (64 output columns after SwiGLU),
// for the down product 128 output columns.  Only the pairs of sixteens of rows
// that the tile really holds are multiplied.  The wide form has eight wavefronts instead of four and 256 weight rows
// (template parameter NWW = 4): per product it moves less through LDS and L2, and it fills a compute unit's LDS alone.
//
// As in moe_mfma.hip the product is formed transposed (A = weight rows,
// B = activation rows), so lane l ends up with four consecutive output
// columns of one row.  The wavefronts are laid out NWW x 2: wavefront
// (wi, xi) owns 64 of the weight rows (for gate|up: 32 gate rows and their up
// rows) and every second sixteen of activation rows, so it reads 4 + 5 operand
// pieces for 20 products.
//
// What bounds it: with few rows per expert the weights (5.8 TB/s with 64 rows of 64 experts of 2,560).  With many the
// products would, but a workgroup's wavefronts meet at every barrier, and what is not laid under the products there
// adds to them.  The reduction runs in stages of 64 through two LDS buffers, and a stage in halves of 32: while a half is
// multiplied, the next half's operands are already on their way from LDS into other registers, also over the end of the
// stage, and the next stage's writes and the loads of the stages after it stand between the products.  One barrier a
// stage, between its halves.  Both products, us, against operands read behind the barrier, each use waited for, and row
// tiles dealt to the dies as wholes: 60 experts of 1,408, rows of 2,048 numbers: 136 rows each 166 + 98 (185 + 104); 23 rows
// and four experts of 340 rows 143 + 77 (169 + 93); one expert of 5,632 with 2,048 rows 109 + 60 (150 + 82).  64 experts of
// 2,560, rows of 3,584, wide: 64 rows each 403 + 241 (406 + 241); with eight experts of 512 rows 543 + 305 (579 + 328), 85
// rows and eight of 682 587 + 348 (684 + 387).  (Weights straight into registers as operands, past LDS: sixteen rows of 64
// bytes a load are half as fast for one compute unit as eight of 128.  One wavefront a SIMD with 512 registers: no better.)
// LDS rows are 128 bytes with their 16-byte pieces permuted, so that operand reads and writes fall on distinct banks.
//
// An expert of up to 64 rows has one tile, and its weights are read once: past the caches (non-temporal, whole lines).  With
// more rows that gains nothing (64 experts of 2,560 with 64 rows on average: 404 us up to 64 rows, 423 up to 96).  Results go through LDS,
// so that a store is 16 bytes a lane of whole lines and not 8 of sixteen rows.  Both products, us, against every load through
// the caches and results straight from the registers: 60 experts of 1,408, rows of 2,048, beside four of every row: 64 rows
// in all 116 + 60 (130 + 68), 340 rows 119 + 67 (134 + 73); 2,048 rows unevenly over the 60 163 + 86 (181 + 98); 64 experts of 2,560, rows of
// 3,584, wide, beside eight of every row: 682 rows 678 + 359 (687 + 372).
//
// Where experts have more rows than a tile (2,048 rows over 60 experts, 137 on average: a third of them), each of an
// expert's row tiles asked for all its weights again, a column block's 20 us after the other tile's: 1.0 GB past L2 for
// 0.69 GB of weights at 6.1 TB/s.  Now they go together (see the kernel): steps of 8 layers and 1,024 / 1,300 / 2,048
// tokens 3,979 / 4,497 / 5,253 -> 3,883 / 4,416 / 5,150 us.
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// the row-tile map is made for tiles of this many rows (the wide form's hold 192)
#define TL_ROWS(NWW) ((NWW) == 2 ? 160 : 192)
#define TL_K 64
// NWW: wavefronts along the weight rows (2 or 4; two along the activation rows): 64 NWW weight rows and 128 NWW
// threads per workgroup.  With four, a row tile's activations are read for half as many column blocks.
#define TL_THREADS(NWW) (128 * (NWW))
#define TL_STRIDE 64  // elements per LDS row: no padding; the eight 16-byte pieces of a row are stored permuted
#define TL_XTILE(NWW) (TL_ROWS(NWW) * TL_STRIDE)  // (staged in steps of 16 NWW rows)
#define TL_WTILE(NWW) (64 * (NWW) * TL_STRIDE)
// piece p of row r lies at piece p ^ ((r >> 1) & 7): the sixteen rows that a quarter of a wavefront reads at one
// piece index then fall on sixteen different groups of four banks, as do the pieces that sixteen lanes write
__device__ __forceinline__ int tl_at(int row, int piece) { return row * TL_STRIDE + ((piece ^ ((row >> 1) & 7)) << 3); }

// One row tile x 64 NWW weight rows.  NP: pairs of sixteens of activation rows the tile holds, one of each a wavefront.
template <bool GATE_UP, int NP, int NWW, bool ONCE>
__device__ __forceinline__ void
tiled_body(const __bf16* a, const __bf16* w, __bf16* out, const int32_t* __restrict__ rows, int n_out, int width,
           int e, int row0, int row_end, int col_block, __bf16* ws, __bf16* xs, int act, float glu_limit) {
  // (a and w are plain pointers on purpose: loads through `const __restrict__` ones may be moved by the
  // optimiser, which sinks them to their first use and so undoes the prefetch)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int wi = wave % NWW, xi = wave / NWW;
  constexpr int STEP = 16 * NWW;                        // rows that the workgroup's threads stage at once
  constexpr int NPX = (32 * NP + STEP - 1) / STEP, NPW = 4;  // pieces per thread and stage
  constexpr int NS = (NWW == 2 ? NP <= 3 : NP <= 4) ? 4 : 2;  // register sets: so many stages are on their way
  constexpr int WROWS = 64 * NWW, HALF = WROWS / 2;
  constexpr int COLS = GATE_UP ? HALF : WROWS;          // output columns of this workgroup
  const int n0 = col_block * COLS;

  const int64_t w_rows = GATE_UP ? 2 * static_cast<int64_t>(n_out) : n_out;
  // (32-bit offsets: the entry point has checked that one expert's weights and the activations stay below 2^31)
  const __bf16* w_expert = w + static_cast<int64_t>(e) * w_rows * width;
  unsigned wsrc[NPW], xsrc[NPX];  // where the rows of this thread's pieces start
#pragma unroll
  for (int i = 0; i < NPW; ++i) {
    const int r = (tid >> 3) + STEP * i;
    const int src_row = GATE_UP ? (r < HALF ? 0 : n_out) + min(n0 + (r % HALF), n_out - 1) : min(n0 + r, n_out - 1);
    wsrc[i] = static_cast<unsigned>(src_row) * static_cast<unsigned>(width);
  }
#pragma unroll
  for (int i = 0; i < NPX; ++i) {
    const int gr = min(row0 + (tid >> 3) + STEP * i, row_end - 1);  // rows past the end repeat the last one; their results are dropped
    xsrc[i] = static_cast<unsigned>(rows ? rows[gr] : gr) * static_cast<unsigned>(width);
  }
  const int dst = tl_at(tid >> 3, tid & 7);  // rows STEP further on have the same permutation

  bf16x8 wreg[NS][NPW], xreg[NS][NPX];
  // Experts walk the reduction in the same order but start at different stages (and wrap round): were all
  // workgroups at the same offset of their weight rows at the same time, a row length that is a power of two
  // would send their loads to the same few memory channels (measured with few rows per expert: 4.0 instead of
  // 5.0 TB/s at rows of 4,096 bytes).  The order of a row's additions depends only on its expert, so results repeat
  // bit for bit; workgroups of one expert stay together (they read the same weights, or the same activations).
  const int stages = (width + TL_K - 1) / TL_K, kspan = stages * TL_K;
  const int rot = (width % 512 == 0)  // rows of a multiple of 1,024 bytes
                      ? static_cast<int>((static_cast<unsigned>(e) * 3u) % static_cast<unsigned>(stages)) * TL_K
                      : 0;
  auto place = [&](int s) {  // where stage s starts in a row (past the end: the last stage again)
    const int k0 = min(s * TL_K, kspan - TL_K);
    return k0 + rot < kspan ? k0 + rot : k0 + rot - kspan;
  };
  // (a piece that does not exist, where the width is no multiple of 64, is the row's last one; zeros take its place)
  auto fetch = [&](int s, int set) {
    const unsigned at = min(place(s) + 8 * (tid & 7), width - 8);
#pragma unroll
    for (int i = 0; i < NPW; ++i) {
      const bf16x8* from = reinterpret_cast<const bf16x8*>(w_expert + (wsrc[i] + at));
      wreg[set][i] = ONCE ? __builtin_nontemporal_load(from) : *from;
    }
#pragma unroll
    for (int i = 0; i < NPX; ++i) xreg[set][i] = *reinterpret_cast<const bf16x8*>(a + (xsrc[i] + at));
  };
  auto stage = [&](int buf, int set) {
#pragma unroll
    for (int i = 0; i < NPW; ++i)
      *reinterpret_cast<bf16x8*>(ws + buf * TL_WTILE(NWW) + dst + STEP * i * TL_STRIDE) = wreg[set][i];
#pragma unroll
    for (int i = 0; i < NPX; ++i)
      *reinterpret_cast<bf16x8*>(xs + buf * TL_XTILE(NWW) + dst + STEP * i * TL_STRIDE) = xreg[set][i];
  };

  f32x4 acc[4][NP];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int t = 0; t < NP; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // this lane's operand pieces: row (sixteen) + m, piece 4 kk + g; the permutation depends on m only
  int xat[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) xat[kk] = tl_at(m, 4 * kk + g);
  const int wrow = (GATE_UP ? 32 : 64) * wi * TL_STRIDE, xrow = 16 * xi * TL_STRIDE;
  struct Half { bf16x8 w[4], x[NP]; };
  Half h0, h1;
  auto read_w = [&](Half& h, int buf, int kk) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // gate|up: blocks 32 wi + {0, 16} and their up rows; down: 64 wi + 16 j
      const int block = GATE_UP ? 16 * (j & 1) + HALF * (j >> 1) : 16 * j;
      h.w[j] = *reinterpret_cast<const bf16x8*>(ws + buf * TL_WTILE(NWW) + wrow + xat[kk] + block * TL_STRIDE);
    }
  };
  auto read_x = [&](Half& h, int buf, int kk) {
#pragma unroll
    for (int t = 0; t < NP; ++t) h.x[t] = *reinterpret_cast<const bf16x8*>(xs + buf * TL_XTILE(NWW) + xrow + xat[kk] + 32 * t * TL_STRIDE);
  };
  auto products = [&](const Half& h) {
#pragma unroll
    for (int t = 0; t < NP; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h.w[j], h.x[t], acc[j][t], 0, 0, 0);
  };

#pragma unroll
  for (int s = 0; s < NS; ++s) {
    fetch(s, s);
    __builtin_amdgcn_sched_barrier(0);
  }
  stage(0, 0);
  __builtin_amdgcn_sched_barrier(0);
  fetch(NS, 0);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  read_w(h0, 0, 0);
  read_x(h0, 0, 0);
  // Stage s is in LDS buffer s & 1, and the operands of its first half are in registers.  While those are multiplied,
  // the second half's are read, stage s + 1 goes from its registers into the other buffer (whose last readers passed the
  // previous barrier) and the registers it leaves take the loads of stage s + 1 + NS.  A barrier; while the second half
  // is multiplied, the first operands of stage s + 1 are read.
#define TL_STAGE(S, B, SET)                                                       \
  {                                                                               \
    stage(1 - (B), ((SET) + 1) % NS);                                             \
    fetch((S) + 1 + NS, ((SET) + 1) % NS);                                        \
    read_w(h1, B, 1);                                                             \
    read_x(h1, B, 1);                                                             \
    products(h0);                                                                 \
    TL_ORDER_A                                                                    \
    __builtin_amdgcn_sched_barrier(0);                                            \
    __syncthreads();                                                              \
    read_w(h0, 1 - (B), 0);                                                       \
    read_x(h0, 1 - (B), 0);                                                       \
    products(h1);                                                                 \
    TL_ORDER_B                                                                    \
    __builtin_amdgcn_sched_barrier(0);                                            \
  }
  // what goes between the products: first half NP + 4 reads, NPW + NPX writes and loads; second half NP + 4 reads
#define TL_ORDER_A                                                                \
  _Pragma("unroll") for (int t = 0; t < NP; ++t) {                                \
    __builtin_amdgcn_sched_group_barrier(0x100, (2 * NP + 3) / NP, 0);      \
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                       \
    __builtin_amdgcn_sched_group_barrier(0x200, (NPW + NPX + NP - 1) / NP, 0);    \
    __builtin_amdgcn_sched_group_barrier(0x020, (NPW + NPX + NP - 1) / NP, 0);    \
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                       \
  }
#define TL_ORDER_B                                                                \
  _Pragma("unroll") for (int t = 0; t < NP; ++t) {                                \
    __builtin_amdgcn_sched_group_barrier(0x100, (2 * NP + 3) / NP, 0);      \
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);                           \
  }
  // Whole turns only, and no way out of a turn's middle: a way out would join the states of the loads of all
  // stages, and the loop's first wait would have to be for the worst of them.  A stage that is not whole is left to
  // the end, too.
  const bool ragged = (width & (TL_K - 1)) != 0;
  const int turns = (stages - (ragged ? 1 : 0)) / NS;
  int s = 0;
  for (int i = 0; i < turns; ++i, s += NS) {
    TL_STAGE(s, 0, 0)
    TL_STAGE(s + 1, 1, 1)
    if constexpr (NS == 4) {
      TL_STAGE(s + 2, 0, 2)
      TL_STAGE(s + 3, 1, 3)
    }
  }
#undef TL_STAGE
#undef TL_ORDER_A
#undef TL_ORDER_B
  const bf16x8 zero = {(__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f,
                       (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f};
  auto last = [&](int at, int i) {  // one of the last stages (at most NS: their operands are all on their way)
    stage(1 - (i & 1), (i + 1) % NS);
    read_w(h1, i & 1, 1);
    read_x(h1, i & 1, 1);
    if (ragged && at == stages - 1) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        if (place(at) + 32 * kk + 8 * g >= width) {
          Half& h = kk ? h1 : h0;
#pragma unroll
          for (int j = 0; j < 4; ++j) h.w[j] = zero;
#pragma unroll
          for (int t = 0; t < NP; ++t) h.x[t] = zero;
        }
    }
    products(h0);
    __syncthreads();
    read_w(h0, 1 - (i & 1), 0);
    read_x(h0, 1 - (i & 1), 0);
    products(h1);
  };
  const int rest = stages - s;
  if (rest > 0) {
    last(s, 0);
    if (rest > 1) {
      last(s + 1, 1);
      if constexpr (NS == 4) {
        if (rest > 2) {
          last(s + 2, 2);
          if (rest > 3) last(s + 3, 3);
        }
      }
    }
  }

  // lane holds weight rows (block) + 4 g + i of activation row row0 + 16 (2 t + xi) + m
  auto result = [&](int t, int j, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = acc[j][t][i];
      if (GATE_UP) v[i] = ix_glu<true>(v[i], acc[GATE_UP ? j + 2 : j][t][i], glu_limit);
      else if (act) v[i] = v[i] > 0.f ? v[i] * v[i] : 0.f;  // the square of relu
    }
  };
  if (((n_out & 7) | static_cast<int>(reinterpret_cast<uintptr_t>(out) & 15)) == 0) {
    // The tile goes through LDS, so that a store is 16 bytes a lane and whole lines.
    constexpr int OUT_STRIDE = COLS + 8;
    static_assert(TL_ROWS(NWW) * OUT_STRIDE <= 2 * (TL_XTILE(NWW) + TL_WTILE(NWW)), "the result's tile fits the stages' LDS");
    __bf16* const tile = ws;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NP; ++t)
#pragma unroll
      for (int j = 0; j < (GATE_UP ? 2 : 4); ++j) {
        float v[4];
        result(t, j, v);
        *reinterpret_cast<bf16x4*>(tile + (16 * (2 * t + xi) + m) * OUT_STRIDE + (GATE_UP ? 32 : 64) * wi + 16 * j + 4 * g) =
            bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
      }
    __syncthreads();
    constexpr int LANES = COLS / 8, AT_ONCE = TL_THREADS(NWW) / LANES;  // lanes of a row; rows that the workgroup stores at once
    const int c = 8 * (tid % LANES);
    if (n0 + c < n_out)
      for (int r = tid / LANES; r < min(32 * NP, row_end - row0); r += AT_ONCE)
        *reinterpret_cast<bf16x8*>(out + static_cast<int64_t>(row0 + r) * n_out + n0 + c) =
            *reinterpret_cast<const bf16x8*>(tile + r * OUT_STRIDE + c);
    return;
  }
  const bool vec = (n_out & 3) == 0;
#pragma unroll
  for (int t = 0; t < NP; ++t) {
    const int r = row0 + 16 * (2 * t + xi) + m;
    if (r >= row_end) continue;
#pragma unroll
    for (int j = 0; j < (GATE_UP ? 2 : 4); ++j) {
      const int nb = n0 + (GATE_UP ? 32 : 64) * wi + 16 * j + 4 * g;
      float v[4];
      result(t, j, v);
      __bf16* dst = out + static_cast<int64_t>(r) * n_out + nb;
      if (nb + 4 <= n_out && vec) {
        bf16x4 o = {(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
        *reinterpret_cast<bf16x4*>(dst) = o;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nb + i < n_out) dst[i] = (__bf16)v[i];
      }
    }
  }
}

template <bool GATE_UP, int NWW>
__global__ void __launch_bounds__(TL_THREADS(NWW)) __attribute__((amdgpu_waves_per_eu(2, 2)))
moe_grouped_tiled_kernel(const __bf16* a, const __bf16* w, __bf16* out, const int32_t* __restrict__ offsets,
                         const int32_t* __restrict__ rows,
                         const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_row0,
                         const int32_t* __restrict__ tile_info, int n_out, int width, int n_col_blocks,
                         int act, float glu_limit, int last_tiles, int last_each) {
  __shared__ __attribute__((aligned(16))) __bf16 ws[2 * (TL_WTILE(NWW) + TL_XTILE(NWW))];
  __bf16* const xs = ws + 2 * TL_WTILE(NWW);
  // Workgroups go to the chip's eight dies in turn, by their number, and each die has its own L2 and its own share of the
  // memory's bandwidth.  The (row tile, column block) pairs, tile by tile, are cut into eight equal runs, one a die, so that
  // the column blocks of a tile, which read the same activations, share an L2 and no die has more of them than another.
  // The last `last_tiles` row tiles are those of experts that every token uses (the shared expert's pieces): full tiles,
  // bound by the matrix cores, where the others hold few rows and wait for their weights.  They are cut by themselves, and
  // a die works them spread evenly among its others, so that at any time some workgroups multiply while the rest keep
  // the memory busy: in runs of as many as a tile has column blocks, and `last_each` tiles of one expert together, column
  // block by column block, as they read the same weights.  (Whole tiles dealt to the dies in turn: some had a tile more,
  // 163 against 103 us at one expert of 2,048 rows, wide; full ones spread one by one: 151 + 84 against 140 + 79 us at 23
  // rows of 60 experts and 340 of four, as the others' weights and activations then leave L2 between uses.)
  const int n_tiles = tile_info[0];
  const unsigned die = blockIdx.x & 7, i = blockIdx.x >> 3;
  const bool spread = last_tiles > 0 && last_tiles < n_tiles;
  const int n_light = spread ? n_tiles - last_tiles : n_tiles;
  const unsigned light = static_cast<unsigned>(n_light) * n_col_blocks;
  const unsigned full = spread ? static_cast<unsigned>(last_tiles) * n_col_blocks : 0u;
  auto cut = [&](unsigned n, unsigned d) { return static_cast<unsigned>(static_cast<uint64_t>(n) * d >> 3); };
  const unsigned light0 = cut(light, die), full0 = cut(full, die);
  const unsigned n_full = cut(full, die + 1) - full0, n_mine = cut(light, die + 1) - light0 + n_full;
  if (i >= n_mine) return;
  bool is_full = false;
  unsigned pair = light0 + i;
  if (n_full > 0) {
    const unsigned run = n_col_blocks, runs = (n_full + run - 1) / run, period = max(n_mine / runs, run);
    const unsigned r = i / period, off = i % period;  // run r starts at place r * period
    const unsigned len = r < runs ? min(run, n_full - r * run) : 0;
    is_full = off < len;
    pair = is_full ? light + full0 + r * run + off : light0 + i - (r < runs ? r * run + len : n_full);
  }
  int tile = static_cast<int>(pair / n_col_blocks), col_block = static_cast<int>(pair % n_col_blocks);
  if (is_full && last_each > 1) {  // (the row tiles of an expert one after the other for a column block)
    const unsigned at = pair - light, per = static_cast<unsigned>(last_each) * n_col_blocks, in = at % per;
    tile = n_tiles - last_tiles + static_cast<int>(at / per * last_each + in % last_each);
    col_block = static_cast<int>(in / last_each);
  }
  const int e = tile_expert[tile];
  int row0 = tile_row0[tile];
  const int row_end = offsets[e + 1], first_row = offsets[e];
  if (!is_full && row_end - first_row > TL_ROWS(NWW)) {
    // Row tiles of an expert that has several read the same weights: up to four of them one after the other for a column
    // block, so that all but the first find the weights in L2.  (Tiles of the expert that are among the last ones have
    // been dealt out above.)
    const int nth = (row0 - first_row) / TL_ROWS(NWW), first = tile - (nth & 3);
    const int of_expert = (row_end - first_row + TL_ROWS(NWW) - 1) / TL_ROWS(NWW) - (nth & ~3);
    const unsigned n_here = min(min(4, of_expert), n_light - first);
    const unsigned in = pair - static_cast<unsigned>(first) * n_col_blocks;
    tile = first + static_cast<int>(in % n_here);
    col_block = static_cast<int>(in / n_here);
    row0 = tile_row0[tile];
  }
  const int held = min(TL_ROWS(NWW), row_end - row0);
  if (held <= 0) return;
  const bool once = held == row_end - first_row && held <= 64;  // an expert's only tile, few rows
#define CALL(NP, ONCE) \
  tiled_body<GATE_UP, NP, NWW, ONCE>(a, w, out, rows, n_out, width, e, row0, row_end, col_block, ws, xs, act, glu_limit)
#define BODY(NP) CALL(NP, false)
  switch ((held + 31) >> 5) {  // pairs of sixteens of rows this tile holds
    case 1: if (once) CALL(1, true); else BODY(1); break;
    case 2: if (once) CALL(2, true); else BODY(2); break;
    case 3: BODY(3); break;
    case 4: BODY(4); break;
    case 5: BODY(5); break;
    default: BODY((NWW == 4 ? 6 : 5)); break;  // (six in the wide form only)
  }
#undef BODY
#undef CALL
}

// The row-tile map must have been made for tiles of 160 rows, for the wide form of 192.  `wide`: see below.
// gate_up: 0 a plain product, 1 gate|up rows with SwiGLU, 2 a plain product whose results pass the square of relu.
// glu_limit > 0: the gate|up rows meet in the clamped form (`ix_glu`).  last_tiles: so many tiles at the end of the
// map are worked spread among the others; `last_each` consecutive ones of them belong to one expert.
extern "C" int ix_moe_grouped_tiled(const void* a, const void* w, void* out, const int32_t* offsets,
                                    const int32_t* rows, const int32_t* tile_expert, const int32_t* tile_row0,
                                    const int32_t* tile_info, int max_tiles, int64_t a_rows, int64_t n_out,
                                    int64_t width, int gate_up, int wide, float glu_limit, int last_tiles, int last_each,
                                    hipStream_t stream) {
  IX_REQUIRE(n_out > 0 && width > 0 && max_tiles >= 0 && last_tiles >= 0 && last_each > 0, "sizes must be positive");
  IX_REQUIRE(last_tiles % last_each == 0, "the last tiles come in equal groups");
  IX_REQUIRE(width % 8 == 0, "the reduction width must be a multiple of 8 for the matrix-core kernel");
  IX_REQUIRE(n_out < (1 << 30) && width < (1 << 30), "sizes too large");
  IX_REQUIRE(a_rows >= 0 && a_rows * width < (int64_t(1) << 31) && (gate_up == 1 ? 2 : 1) * n_out * width < (int64_t(1) << 31),
             "the activations, and one expert's weights, must hold fewer than 2^31 numbers");
  IX_REQUIRE(max_tiles <= 65535, "too many row tiles for one launch");
  if (max_tiles == 0) return 0;
  // wide: four wavefronts along the weight rows instead of two (256 weight rows per workgroup, 112 KB of LDS, one
  // workgroup per compute unit): the activations are staged for half as many column blocks.  Same sums in the
  // same order either way.
  const int nww = wide ? 4 : 2;
  const int cols = gate_up == 1 ? 32 * nww : 64 * nww;
  const int n_col_blocks = static_cast<int>((n_out + cols - 1) / cols);
  const int64_t groups = 8 * (static_cast<int64_t>(n_col_blocks) * max_tiles / 8 + 2);  // (a die has at most this many pairs)
  IX_REQUIRE(groups < (int64_t(1) << 31), "too many workgroups for one launch");
  dim3 grid(static_cast<unsigned>(groups)), block(TL_THREADS(nww));
#define LAUNCH(GU, NWW)                                                                                             \
  hipLaunchKernelGGL((moe_grouped_tiled_kernel<GU, NWW>), grid, block, 0, stream, (const __bf16*)a, (const __bf16*)w, \
                     (__bf16*)out, offsets, rows, tile_expert, tile_row0, tile_info, (int)n_out, (int)width,         \
                     n_col_blocks, gate_up == 2 ? 1 : 0, glu_limit, std::min(last_tiles, max_tiles), last_each)
  if (nww == 4) {
    if (gate_up == 1) LAUNCH(true, 4);
    else LAUNCH(false, 4);
  } else {
    if (gate_up == 1) LAUNCH(true, 2);
    else LAUNCH(false, 2);
  }
#undef LAUNCH
  return ix_check_launch("ix_moe_grouped_tiled");
}
