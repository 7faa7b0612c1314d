// The order in which the float32 grouped products' workgroups work the row tiles of the grouping kernel's map.
#pragma once

#include "common.h"

#define TF_ROWS 64  // rows of a tile of the map

// The tiles with most rows come first, so that what is left at the end is short (and a tile's column blocks go to the
// chip's eight dies in turn, so that each has as much of it; a die's run of whole tiles took 133 to 178 us at 511 tokens).  Tiles of as
// many sixteens stay together in the map's order; beyond 512 of them the end no longer matters.  (Long and short tiles in
// turn leave half the chip idle at times: workgroups are handed out in order, each to a place of its own.)
// -> the tile at place `tile`; the same for all lanes of a wavefront, all of them at work.
__device__ __forceinline__ int tf_tile(int tile, int n_tiles, const int32_t* offsets, const int32_t* tile_expert, const int32_t* tile_row0) {
  if (n_tiles > 8 * 64) return tile;
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
  return __builtin_amdgcn_readfirstlane(tile);
}
