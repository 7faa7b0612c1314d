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
// What bounds it: with few rows per expert the weights, with many the products; in between each waits for the other
// in turn.  The reduction runs in stages of 64 through a ring of LDS buffers that the loads fill by themselves
// (`global_load_lds`, 16 bytes a lane; which piece a lane asks for makes the permutation below): no register holds a
// piece on its way and no wavefront writes LDS.  (With the pieces through registers, products and operand reads alone
// ran at 1,580 TFLOP/s, with the writes 1,170, with the loads 950.)  A stage goes in halves of 32: while a half is
// multiplied, the next half's operands are read from LDS into other registers, also over the end of the stage.  One
// barrier a stage, between its halves: behind it stage s + 1 has landed for everybody and everybody is done with the
// buffers of stage s, which take the loads of the stages after those that are on their way (`Ring`).
//   The rings: what LDS holds, the weights, which come from memory, at least as deep as the activations, which come from
// L2.  (Four against three stages for tiles of up to 64 rows: no difference; two: 484 against 412 us at 64 experts of 2,560,
// rows of 3,584, 64 rows each on average.)
//   A launch of no more narrow workgroups than compute units gives each all of the LDS: three stages of the highest tiles too, of which
// half of it holds two, and six of the lowest.  Eight experts of 768 on a width of 2,048, 203 tokens of six, both products 36 + 16 us with half,
// so 29.4 + 13.9 (with the pieces through registers 28.4 + 13.7); four of 2,048 on 2,816, 359 tokens 50 + 34, so 39.5 + 27.6 (35.7 +
// 23.2).  Four to eight stages are no faster.  Of more workgroups some wait for places: 304 + 304 of them 64 us with half, 96 so.
//   Both products, us, against the pieces through registers: 60 experts of 1,408, rows of 2,048, beside four of every row,
// 340 rows: narrow 128 + 76 (135 + 80), wide 123 + 77 (130 + 83); 2,048 rows unevenly over the 60: wide 166 + 88 (182 + 100);
// 64 experts of 2,560, rows of 3,584, wide, beside eight of every row: 512 rows 524 + 291 (570 + 316), 682 rows 581 + 326 (607
// + 351).  Eight experts of 1,920 rows: 1,080 TFLOP/s (970); the library's dense products 1,080.
//   Built and left out: four wavefronts with 512 registers each and 128 weight rows (a third fewer operand reads; nobody to
// multiply while one waits: 256 against 238 us for eight experts of 512 rows).
// LDS rows are 128 bytes with their 16-byte pieces permuted, so that operand reads fall on distinct banks.
//
// An expert with one tile has its weights read once: past the caches (non-temporal, whole lines; a plain read of memory gives
// 7.0 TB/s that way and 6.1 through them).  2,048 rows unevenly over 60 experts 254 against 268 us for both products.  Weights
// that several tiles read stay cached (2,048 rows 289 us past the caches), and so do those whose rows are no whole lines: rows and stages
// share some, which would come from memory for each of them (128 experts of 656 on 2,920, 513 tokens of four, both products 361 us past the
// caches, 315 through them).  Results go through LDS, so that a store is 16
// bytes a lane of whole lines and not 8 of sixteen rows.
//
// Where experts have more rows than a tile, each of an expert's row tiles would ask for all its weights again, a column
// block's 20 us after the other tile's: they go together (see the kernel).
//
// Operands that do not lie on 16-byte boundaries (`DIRECT` false) go through registers, one piece after the other.
#include <type_traits>

#include "moe_tiled.h"

// Workgroups go to the chip's eight dies in turn, by their number, and each die has its own L2 and its own share of the
// memory's bandwidth.  The (row tile, column block) pairs, tile by tile, are cut into eight equal runs, one a die, so that
// the column blocks of a tile, which read the same activations, share an L2 and no die has more of them than another.
// The last `last_tiles` row tiles are those of experts that every token uses (the shared expert's pieces): full tiles,
// bound by the matrix cores, where the others hold few rows and wait for their weights.  They are cut by themselves, and
// a die works them spread evenly among its others, so that at any time some workgroups multiply while the rest keep
// the memory busy: `last_each` tiles of one expert together for a column block, as they read the same weights, and two
// column blocks a run.  Both products, us, with runs of one block, two, four and all of a tile's: 64 experts of 2,560, rows of
// 3,584, beside eight of every row: 512 rows 810, 827, 832, 852, 682 rows 897, 902, 909, 906; 60 of 1,408, rows of 2,048,
// beside four: 100 rows 180, 174, 172, 172, 340 rows 209, 208, 208, 212.  (Whole tiles dealt to the dies in turn: some
// had a tile more, 163 against 103 us at one expert of 2,048 rows, wide.)
// A second product's tiles are worked as the last ones: as many row tiles of one expert.
template <bool GATE_UP, int NWW>
struct TileList {
  static constexpr int ROWS = TL_ROWS(NWW), COLS = (GATE_UP ? 32 : 64) * NWW;
  const int32_t *offsets, *tile_expert, *tile_row0;
  int n_tiles, n_light, last_tiles, last_each, n_col_blocks, second_rows;
  bool second_first;
  unsigned light, light0, full0, n_full, n;  // n: how many pairs the die has

  struct Pair {
    int e, first_row, row0, row_end, col_block;  // rows row0 to min(row0 + ROWS, row_end) of the expert that starts at first_row
    bool full, second;                           // of the last tiles; of the second product (e 0)
  };

  __device__ __forceinline__ TileList(unsigned die, const int32_t* offsets_, const int32_t* tile_expert_, const int32_t* tile_row0_,
                                      const int32_t* tile_info, int n_col_blocks_, int width, int last_tiles_, int last_each_,
                                      const Second& second)
      : offsets(offsets_), tile_expert(tile_expert_), tile_row0(tile_row0_), n_tiles(tile_info[0]), last_tiles(last_tiles_),
        last_each(last_each_), n_col_blocks(n_col_blocks_), second_rows(second.rows) {
    const bool two = NWW == 4 && second.rows > 0, spread = !two && last_tiles > 0 && last_tiles < n_tiles;
    if (two) last_each = (second.rows + ROWS - 1) / ROWS;
    n_light = spread ? n_tiles - last_tiles : n_tiles;
    light = static_cast<unsigned>(n_light) * n_col_blocks;
    const unsigned full = two ? static_cast<unsigned>(last_each) * ((second.n_out + COLS - 1) / COLS)
                              : spread ? static_cast<unsigned>(last_tiles) * n_col_blocks : 0u;
    auto cut = [&](unsigned pairs, unsigned d) { return static_cast<unsigned>(static_cast<uint64_t>(pairs) * d >> 3); };
    light0 = cut(light, die);
    full0 = cut(full, die);
    n_full = cut(full, die + 1) - full0;
    n = cut(light, die + 1) - light0 + n_full;
    second_first = two && second.width > width;
  }

  // the i-th pair of the die, i < n
  __device__ __forceinline__ Pair pair(unsigned i) const {
    Pair p;
    p.full = false;
    unsigned at = light0 + i;
    if (second_first) {
      // longer ones first: they then end with the others (88 of 88 stages beside some 600 of 22, of 256 places)
      p.full = i < n_full;
      at = p.full ? light + full0 + i : light0 + i - n_full;
    } else if (n_full > 0) {
      const unsigned run = 2u * last_each, runs = (n_full + run - 1) / run, period = max(n / runs, run);
      const unsigned r = i / period, off = i % period;  // run r starts at place r * period
      const unsigned len = r < runs ? min(run, n_full - r * run) : 0;
      p.full = off < len;
      at = p.full ? light + full0 + r * run + off : light0 + i - (r < runs ? r * run + len : n_full);
    }
    p.second = p.full && NWW == 4 && second_rows > 0;
    if (p.second) {
      const int in = static_cast<int>(at - light);
      p.e = 0;
      p.first_row = 0;
      p.row0 = ROWS * (in % last_each);
      p.col_block = in / last_each;
      p.row_end = second_rows;
      return p;
    }
    int tile = static_cast<int>(at / n_col_blocks);
    p.col_block = static_cast<int>(at % n_col_blocks);
    if (p.full && last_each > 1) {  // (the row tiles of an expert one after the other for a column block)
      const unsigned of_last = at - light, per = static_cast<unsigned>(last_each) * n_col_blocks, in = of_last % per;
      tile = n_tiles - last_tiles + static_cast<int>(of_last / per * last_each + in % last_each);
      p.col_block = static_cast<int>(in / last_each);
    }
    p.e = tile_expert[tile];
    p.row0 = tile_row0[tile];
    p.row_end = offsets[p.e + 1];
    p.first_row = offsets[p.e];
    if (!p.full && p.row_end - p.first_row > ROWS) {
      // Row tiles of an expert that has several read the same weights: up to four of them one after the other for a column
      // block, so that all but the first find the weights in L2.  (Tiles of the expert that are among the last ones have
      // been dealt out above.)
      const int nth = (p.row0 - p.first_row) / ROWS, first = tile - (nth & 3);
      const int of_expert = (p.row_end - p.first_row + ROWS - 1) / ROWS - (nth & ~3);
      const unsigned n_here = min(min(4, of_expert), n_light - first);
      const unsigned in = at - static_cast<unsigned>(first) * n_col_blocks;
      tile = first + static_cast<int>(in % n_here);
      p.col_block = static_cast<int>(in / n_here);
      p.row0 = tile_row0[tile];
    }
    return p;
  }
};

#define TL_LDS(ALL) ((ALL) ? 163840 : 81920)  // bytes: all of a compute unit's, or half

// 16 bytes a lane from base + offset to lds + dst + 16 lane, straight or, from anywhere, through registers.
template <bool NT, bool DIRECT>
__device__ __forceinline__ void to_lds(__bf16* lds, unsigned dst, unsigned offset, const void* base) {
  if constexpr (DIRECT) {
    lds_load16<NT>(lds, dst, offset, base);
  } else {
    typedef __bf16 anywhere __attribute__((ext_vector_type(8), aligned(2)));
    const anywhere v = *reinterpret_cast<const anywhere*>(static_cast<const char*>(base) + offset);
    *reinterpret_cast<bf16x8*>(reinterpret_cast<char*>(lds) + dst + 16 * (threadIdx.x & 63)) = v;
  }
}

// How many stages' weights (W) and activations (X) LDS holds.
// ALL: a workgroup has all of a compute unit's LDS.
template <int NP, int NWW, bool ALL> struct Ring {
  static constexpr int XROWS = NWW == 4 ? 64 * ((NP + 1) / 2) : 32 * NP;  // rows staged: whole loads for every wavefront
  static constexpr int NARROW_ALL = NP == 1 ? 6 : NP == 2 ? 4 : 3;
  static constexpr int W = NWW == 4 ? (NP <= 2 ? 4 : 3) : ALL ? NARROW_ALL : (NP == 1 ? 4 : NP <= 4 ? 3 : 2);
  static constexpr int X = NWW == 4 ? (NP <= 2 ? 4 : NP <= 4 ? 3 : 2) : ALL ? NARROW_ALL : (NP == 1 ? 4 : NP == 2 ? 3 : 2);
  static_assert((W * 64 * NWW + X * XROWS) * 2 * TL_STRIDE <= TL_LDS(ALL), "the rings fit");
  static_assert(W == X || W == X + 1, "the waits below count on it");
};

// One row tile x 64 NWW weight rows.  NP: pairs of sixteens of activation rows the tile holds, one of each a wavefront.
template <bool GATE_UP, int NP, int NWW, bool ALL, bool ONCE, bool DIRECT>
__device__ __forceinline__ void
tiled_body(const __bf16* a, const __bf16* w, __bf16* out, const int32_t* __restrict__ rows, int n_out, int width,
           int e, int row0, int row_end, int col_block, __bf16* lds, int act, float glu_limit) {
  using R = Ring<NP, NWW, ALL>;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int wi = wave % NWW, xi = wave / NWW;
  constexpr int WAVES = 2 * NWW, WROWS = 64 * NWW, HALF = WROWS / 2;
  constexpr int NPW = WROWS / 8 / WAVES, NPX = R::XROWS / 8 / WAVES;  // loads of a wavefront a stage, eight rows each
  constexpr int COLS = GATE_UP ? HALF : WROWS;                        // output columns of this workgroup
  constexpr unsigned WT = WROWS * 2 * TL_STRIDE, XT = R::XROWS * 2 * TL_STRIDE;  // bytes of a stage
  const int n0 = col_block * COLS;

  const int64_t w_rows = GATE_UP ? 2 * static_cast<int64_t>(n_out) : n_out;
  // (32-bit offsets: the entry point has checked that one expert's weights and the activations stay below 2^32 bytes)
  const __bf16* w_expert = w + static_cast<int64_t>(e) * w_rows * width;
  unsigned wsrc[NPW], xsrc[NPX];  // where this lane's rows start, in bytes: a wavefront brings rows 8 (wave + WAVES i) to + 7
#pragma unroll
  for (int i = 0; i < NPW; ++i) {
    const int r = 8 * (wave + WAVES * i) + (lane >> 3);
    const int src_row = GATE_UP ? (r < HALF ? 0 : n_out) + min(n0 + (r % HALF), n_out - 1) : min(n0 + r, n_out - 1);
    wsrc[i] = 2u * static_cast<unsigned>(src_row) * static_cast<unsigned>(width);
  }
#pragma unroll
  for (int i = 0; i < NPX; ++i) {
    const int gr = min(row0 + 8 * (wave + WAVES * i) + (lane >> 3), row_end - 1);  // rows past the end repeat the last one; their results are dropped
    xsrc[i] = 2u * static_cast<unsigned>(rows ? rows[gr] : gr) * static_cast<unsigned>(width);
  }
  // The lane's place in its row is piece lane & 7; what belongs there by `tl_at` (the number of a wavefront's eights of rows
  // is as odd or even as the wavefront's own):
  static_assert(WAVES % 2 == 0, "as odd or even");
  const int piece = 8 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4)));

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
  auto at = [&](int s) { return 2u * static_cast<unsigned>(min(place(s) + piece, width - 8)); };
  auto load_w = [&](unsigned buf, int i, unsigned from) {
    to_lds<ONCE, DIRECT>(lds, buf + 1024 * (wave + WAVES * i), wsrc[i] + from, w_expert);
  };
  auto load_x = [&](unsigned buf, int i, unsigned from) {
    to_lds<false, DIRECT>(lds, R::W * WT + buf + 1024 * (wave + WAVES * i), xsrc[i] + from, a);
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
  const __bf16* const ws = lds + (GATE_UP ? 32 : 64) * wi * TL_STRIDE;
  const __bf16* const xs = lds + R::W * WT / 2 + 16 * xi * TL_STRIDE;
  struct Half { bf16x8 w[4], x[NP]; };
  Half h0, h1;
  auto read = [&](Half& h, int i, unsigned wbuf, unsigned xbuf, int kk) {  // the i-th of a half's NP + 4 pieces
    if (i < 4) {  // gate|up: blocks 32 wi + {0, 16} and their up rows; down: 64 wi + 16 j
      const int block = GATE_UP ? 16 * (i & 1) + HALF * (i >> 1) : 16 * i;
      h.w[i] = *reinterpret_cast<const bf16x8*>(ws + wbuf / 2 + xat[kk] + block * TL_STRIDE);
    } else if (i < NP + 4) {
      h.x[i - 4] = *reinterpret_cast<const bf16x8*>(xs + xbuf / 2 + xat[kk] + 32 * (i - 4) * TL_STRIDE);
    }
  };
  auto products = [&](const Half& h, int t) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h.w[j], h.x[t], acc[j][t], 0, 0, 0);
  };

#pragma unroll
  for (int s = 0; s < R::W; ++s) {
    const unsigned from = at(s);
    if (s < R::X)
#pragma unroll
      for (int i = 0; i < NPX; ++i) load_x(s * XT, i, from);
#pragma unroll
    for (int i = 0; i < NPW; ++i) load_w(s * WT, i, from);
  }
  wait_loads<NPW * (R::W - 1) + NPX * (R::X - 1)>();
  lds_barrier();
  unsigned wbuf = 0, xbuf = 0;  // where the present stage lies in the rings
#pragma unroll
  for (int i = 0; i < NP + 4; ++i) read(h0, i, wbuf, xbuf, 0);

  // Stage s, the operands of its first half in registers; LEFT: at least so many stages follow.  Reads and loads go between
  // the products, as many a step as leave the last ones time to arrive.
  constexpr int READS = NP > 1 ? (NP + 4 + NP - 2) / (NP - 1) : 5, LOADS = (NPW + NPX + NP - 1) / NP;
  auto stage = [&](auto left, int s) {
    constexpr int LEFT = decltype(left)::value;
#pragma unroll
    for (int t = 0; t < NP; ++t) {
      if constexpr (LEFT > 0) products(h0, t);
#pragma unroll
      for (int i = READS * t; i < READS * (t + 1); ++i) read(h1, i, wbuf, xbuf, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LEFT == 0) {
      if (width & (TL_K - 1)) {  // the last stage is not whole
        const bf16x8 zero = {(__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f,
                             (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
          if (place(s) + 32 * kk + 8 * g >= width) {
            Half& h = kk ? h1 : h0;
#pragma unroll
            for (int j = 0; j < 4; ++j) h.w[j] = zero;
#pragma unroll
            for (int t = 0; t < NP; ++t) h.x[t] = zero;
          }
      }
#pragma unroll
      for (int t = 0; t < NP; ++t) products(h0, t);
#pragma unroll
      for (int t = 0; t < NP; ++t) products(h1, t);
    } else {
      // Stage s + 1 must have landed.  After its last load there were issued (an iteration issues activations first) the
      // weights of stages up to s + W - 1 and the activations of stages up to s + X - 1, as far as there are so many.
      constexpr int LATER_W = R::W - 2 < LEFT - 1 ? R::W - 2 : LEFT - 1, LATER_X = R::X - 2 < LEFT - 1 ? R::X - 2 : LEFT - 1;
      wait_loads<NPW * LATER_W + NPX * LATER_X>();
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
      const unsigned wfree = wbuf, xfree = xbuf;  // nobody reads stage s any more
      wbuf = wbuf + WT == R::W * WT ? 0 : wbuf + WT;
      xbuf = xbuf + XT == R::X * XT ? 0 : xbuf + XT;
      const unsigned from_x = LEFT >= R::X ? at(s + R::X) : 0u, from_w = LEFT >= R::W ? at(s + R::W) : 0u;
#pragma unroll
      for (int t = 0; t < NP; ++t) {
        products(h1, t);
#pragma unroll
        for (int i = READS * t; i < READS * (t + 1); ++i) read(h0, i, wbuf, xbuf, 0);
#pragma unroll
        for (int i = LOADS * t; i < LOADS * (t + 1); ++i) {
          if (i < NPX) {
            if constexpr (LEFT >= R::X) load_x(xfree, i, from_x);
          } else if (i < NPX + NPW) {
            if constexpr (LEFT >= R::W) load_w(wfree, i - NPX, from_w);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
#define TL_STAGE(LEFT, S) stage(std::integral_constant<int, (LEFT)>{}, (S))
  for (int s = 0; s < stages - R::W; ++s) TL_STAGE(R::W, s);
  if constexpr (R::W > 5)
    if (stages > 5) TL_STAGE(5, stages - 6);
  if constexpr (R::W > 4)
    if (stages > 4) TL_STAGE(4, stages - 5);
  if constexpr (R::W > 3)
    if (stages > 3) TL_STAGE(3, stages - 4);
  if constexpr (R::W > 2)
    if (stages > 2) TL_STAGE(2, stages - 3);
  if (stages > 1) TL_STAGE(1, stages - 2);
  TL_STAGE(0, stages - 1);
#undef TL_STAGE
  wait_loads<0>();  // (with fewer stages than the rings hold, the last one again)

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
    static_assert(TL_ROWS(NWW) * OUT_STRIDE * 2 <= TL_LDS(ALL), "the result's tile fits the stages' LDS");
    __bf16* const tile = lds;
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

template <bool GATE_UP, int NWW, bool ALL, bool DIRECT>
__global__ void __launch_bounds__(TL_THREADS(NWW)) __attribute__((amdgpu_waves_per_eu(2, 2)))
moe_grouped_tiled_kernel(const __bf16* a, const __bf16* w, __bf16* out, const int32_t* __restrict__ offsets,
                         const int32_t* __restrict__ rows,
                         const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_row0,
                         const int32_t* __restrict__ tile_info, int n_out, int width, int n_col_blocks,
                         int act, float glu_limit, int last_tiles, int last_each, Second second) {
  __shared__ __attribute__((aligned(1024))) __bf16 lds[TL_LDS(ALL) / 2];
  const TileList<GATE_UP, NWW> list(blockIdx.x & 7, offsets, tile_expert, tile_row0, tile_info, n_col_blocks, width, last_tiles,
                                    last_each, second);
  const unsigned i = blockIdx.x >> 3;
  if (i >= list.n) return;
  const auto p = list.pair(i);
  const int e = p.e, row0 = p.row0, row_end = p.row_end, col_block = p.col_block;
  // An expert's only tile.  (Rows that are no whole lines share some, which would come from memory for each of them.)
  const bool once = DIRECT && !p.second && row_end - p.first_row <= TL_ROWS(NWW) &&
                    ((width & 63) | static_cast<int>(reinterpret_cast<uintptr_t>(w) & 127)) == 0;
  if (p.second)
    a = second.a, w = second.w, out = second.out, rows = nullptr, n_out = second.n_out, width = second.width, act = 0;
  const int held = min(TL_ROWS(NWW), row_end - row0);
  if (held <= 0) return;
#define CALL(NP, ONCE) \
  tiled_body<GATE_UP, NP, NWW, ALL, ONCE, DIRECT>(a, w, out, rows, n_out, width, e, row0, row_end, col_block, lds, act, glu_limit)
#define BODY(NP) if (once) CALL(NP, DIRECT); else CALL(NP, false)
  switch ((held + 31) >> 5) {  // pairs of sixteens of rows this tile holds
    case 1: BODY(1); break;
    case 2: BODY(2); break;
    case 3: BODY(3); break;
    case 4: BODY(4); break;
    case 5: BODY(5); break;
    default: BODY((NWW == 4 ? 6 : 5)); break;  // (six in the wide form only)
  }
#undef BODY
#undef CALL
}

// The row-tile map must have been made for tiles of 160 rows, for the wide form of 192.  form: 0 narrow; 1 wide, four wavefronts
// along the weight rows instead of two (256 weight rows a workgroup, all of a compute unit's LDS): the activations are staged for half as
// many column blocks; 2 narrow with all of a compute unit's LDS, for launches that leave no two workgroups to a compute unit.
// Same sums in the same order in all of them.
// gate_up: 0 a plain product, 1 gate|up rows with SwiGLU, 2 a plain product whose results pass the square of relu.
// glu_limit > 0: the gate|up rows meet in the clamped form (`ix_glu`).  last_tiles: so many tiles at the end of the
// map are worked spread among the others; `last_each` consecutive ones of them belong to one expert.  a2, w2, out2 (rows2 0: none, and
// with the wide form only): a product of its own in the same launch, out2 [rows2, n_out2] = a2 [rows2, width2] . w2^T, gate|up
// as the grouped one; no last tiles then.  queue (or null): eight counters that hold 0, and the number of tiles of experts with more
// than 128 rows, which the map lists first; with them and the tiles as `ix_moe_dispatch` leaves them behind its queues the wide form may
// be worked by workgroups that stay (moe_tiled_queue.hip).
int ix_moe_grouped_queue(const void* a, const void* w, void* out, const int32_t* rows, const int32_t* tile_info, const void* tiles,
                         int32_t* queue, int max_tiles, int64_t n_out, int64_t width, int gate_up, float glu_limit, const void* a2,
                         const void* w2, void* out2, int64_t rows2, int64_t n_out2, int64_t width2, hipStream_t stream);
extern "C" int ix_moe_grouped_tiled(const void* a, const void* w, void* out, const int32_t* offsets,
                                    const int32_t* rows, const int32_t* tile_expert, const int32_t* tile_row0,
                                    const int32_t* tile_info, int max_tiles, int64_t a_rows, int64_t n_out,
                                    int64_t width, int gate_up, int form, float glu_limit, int last_tiles, int last_each,
                                    const void* a2, const void* w2, void* out2, int64_t rows2, int64_t n_out2,
                                    int64_t width2, int32_t* queue, const void* tiles, hipStream_t stream) {
  IX_REQUIRE(n_out > 0 && width > 0 && max_tiles >= 0 && last_tiles >= 0 && last_each > 0, "sizes must be positive");
  IX_REQUIRE(last_tiles % last_each == 0, "the last tiles come in equal groups");
  IX_REQUIRE(width % 8 == 0, "the reduction width must be a multiple of 8 for the matrix-core kernel");
  IX_REQUIRE(n_out < (1 << 30) && width < (1 << 30), "sizes too large");
  IX_REQUIRE(a_rows >= 0 && a_rows * width < (int64_t(1) << 31) && (gate_up == 1 ? 2 : 1) * n_out * width < (int64_t(1) << 31),
             "the activations, and one expert's weights, must hold fewer than 2^31 numbers");
  IX_REQUIRE(max_tiles <= 65535, "too many row tiles for one launch");
  IX_REQUIRE(form >= 0 && form <= 2, "form must be 0, 1 or 2");
  IX_REQUIRE(rows2 >= 0 && (rows2 == 0 || (form == 1 && last_tiles == 0 && gate_up != 2 && n_out2 > 0 && width2 > 0)),
             "a second product needs the wide form, no last tiles and positive sizes");
  IX_REQUIRE(width2 % 8 == 0 || rows2 == 0, "the reduction width must be a multiple of 8 for the matrix-core kernel");
  IX_REQUIRE(rows2 == 0 || (n_out2 < (1 << 30) && width2 < (1 << 30) && rows2 * width2 < (int64_t(1) << 31) &&
                            (gate_up == 1 ? 2 : 1) * n_out2 * width2 < (int64_t(1) << 31)),
             "the second product's activations, and its weights, must hold fewer than 2^31 numbers");
  if (max_tiles == 0 && rows2 == 0) return 0;
  const int nww = form == 1 ? 4 : 2;
  const int cols = gate_up == 1 ? 32 * nww : 64 * nww;
  const int n_col_blocks = static_cast<int>((n_out + cols - 1) / cols);
  const int64_t full2 = rows2 == 0 ? 0 : (rows2 + TL_ROWS(4) - 1) / TL_ROWS(4) * ((n_out2 + cols - 1) / cols);
  const int64_t groups = 8 * ((static_cast<int64_t>(n_col_blocks) * max_tiles + full2) / 8 + 2);  // (a die has at most this many pairs)
  IX_REQUIRE(groups < (int64_t(1) << 31), "too many workgroups for one launch");
  if (form == 1 && queue && tiles) {
    const int rc = ix_moe_grouped_queue(a, w, out, rows, tile_info, tiles, queue, max_tiles, n_out, width, gate_up, glu_limit, a2, w2,
                                        out2, rows2, n_out2, width2, stream);
    if (rc != 2) return rc;
  }
  dim3 grid(static_cast<unsigned>(groups)), block(TL_THREADS(nww));
  const uintptr_t second = rows2 == 0 ? 0 : reinterpret_cast<uintptr_t>(a2) | reinterpret_cast<uintptr_t>(w2);
  const bool direct = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w) | second) & 15) == 0;
#define LAUNCH(GU, NWW, ALL, DIRECT)                                                                                     \
  hipLaunchKernelGGL((moe_grouped_tiled_kernel<GU, NWW, ALL, DIRECT>), grid, block, 0, stream, (const __bf16*)a,         \
                     (const __bf16*)w, (__bf16*)out, offsets, rows, tile_expert, tile_row0, tile_info, (int)n_out,  \
                     (int)width, n_col_blocks, gate_up == 2 ? 1 : 0, glu_limit, std::min(last_tiles, max_tiles), last_each,         \
                     (Second{(const __bf16*)a2, (const __bf16*)w2, (__bf16*)out2, (int)rows2, (int)n_out2, (int)width2}))
#define FORM(GU)                                       \
  if (form == 1 && direct) LAUNCH(GU, 4, true, true);  \
  else if (form == 1) LAUNCH(GU, 4, true, false);      \
  else if (!direct) LAUNCH(GU, 2, false, false);       \
  else if (form == 2) LAUNCH(GU, 2, true, true);       \
  else LAUNCH(GU, 2, false, true)
  if (gate_up == 1) {
    FORM(true);
  } else {
    FORM(false);
  }
#undef FORM
#undef LAUNCH
  return ix_check_launch("ix_moe_grouped_tiled");
}
