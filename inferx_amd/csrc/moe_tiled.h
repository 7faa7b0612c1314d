// What the two kernels of the grouped products in tiles share: sizes of a tile, places in LDS, a second product.
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
