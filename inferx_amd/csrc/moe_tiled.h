// What the two kernels of the grouped products in tiles share: sizes of a tile, places in LDS, and which (row tile, column
// block) pair a workgroup of a die works when.
#pragma once

#include "lds_loads.h"

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
// piece p of row r lies at piece p ^ ((r >> 1) & 7): the sixteen rows that a quarter of a wavefront reads at one
// piece index then fall on sixteen different groups of four banks
__device__ __forceinline__ int tl_at(int row, int piece) { return row * TL_STRIDE + ((piece ^ ((row >> 1) & 7)) << 3); }

// A second product of the launch: out [rows, n_out] = a [rows, width] . w^T, one set of weights for all rows (with gate|up the two
// sets of n_out rows).  rows 0: none.
struct Second {
  const __bf16 *a, *w;
  __bf16* out;
  int rows, n_out, width;
};

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
