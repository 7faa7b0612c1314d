// The wide form of the grouped expert products in tiles (moe_tiled.hip) by workgroups that stay: as many as there are compute
// units, each takes the next (row tile, column block) pair of its die from a counter until none is left.  Same tiles, same sums in
// the same order.
//
// What it is for: with a workgroup for each pair, a pair of 43 us (192 rows, 256 weight rows, a reduction of 2,048) spent 3.3 us on its
// tables, row numbers and first loads, 5.8 behind its last product, and its place was empty for 2.2 before the next one had
// it.  A workgroup that stays takes its next pair from the counter shortly before the end: when the last stage has landed, the weights of
// the next pair's first two stages follow it in the ring, with the row numbers, and behind the last operand
// read everything else of the next pair's start is asked for, so that the results are formed and stored while it arrives.
// By time stamps a pair takes 26 to 40 us now of the 29 to 45 from one start on a place to the next; the rest of it is the reduction, which the
// memory's rate bounds for few rows and the card's power for many.  Gate|up + down in a step, a workgroup for each pair -> so: 2,048 tokens in 60
// experts of 1,408 beside a shared one 261 + 135 -> 247 + 130 us, 340 tokens beside four pieces 127 + 76 -> 122 + 72; 64 experts of 2,560
// beside eight pieces, 512 tokens 547 + 305 -> 520 + 297, 682 tokens 603 + 341 -> 588 + 334.  Pairs dealt out beforehand, every 32nd to
// a workgroup, instead of from a counter would lose most of that: they take 27 to 100 us.  Taken at the start of the pair before
// instead of at its end, the next pair waited behind one of 100 us while other places were empty (down 126 -> 134 us).
//
// LDS: three stages of weights (32 KB each), two or three of activations, the row numbers of the next pair, the tiles, and the die's
// list of pairs, which every workgroup makes for itself while its first loads are on their way.
//
// The counts of loads that the waits name rest on their order: loads, stores and the counter's atomic of a wavefront are all
// done in the order in which they were issued.
#include <type_traits>

#include "moe_tiled.h"

#define TQ_PLACES 256                                // workgroups: one a compute unit, an eighth of them a die
#define TQ_W 3                                       // stages of weights in LDS
#define TQ_THREADS TL_THREADS(4)
#define TQ_LDS 163840
#define TQ_WT (256 * 2 * TL_STRIDE)                  // bytes of a stage's weights
#define TQ_X_AT (TQ_W * TQ_WT)                       // bytes: where the activations start
#define TQ_X_BYTES 49152
#define TQ_ROWS_AT (TQ_X_AT + TQ_X_BYTES)            // row numbers, 64 of a wavefront
#define TQ_NEXT_AT (TQ_ROWS_AT + 8 * 256)            // the next pair's place in the list
#define TQ_TILES_AT (TQ_NEXT_AT + 16)                // the tiles: 8 bytes each
#define TQ_TILES 768                                 // ... so many
#define TQ_LIST_AT (TQ_TILES_AT + 8 * TQ_TILES)      // the list: 4 bytes a pair
#define TQ_LIST 1536                                 // ... of so many
static_assert(TQ_LIST_AT + 4 * TQ_LIST <= TQ_LDS, "everything fits LDS");
#define TQ_SECOND 32768  // bit of a list's entry: of the second product
#define TQ_USED (1 << 30)  // bit of a counter: a launch has been worked by it (and it is at its start again)

// Activations of a tile of NP pairs of sixteens of rows.  (LOADS: of a wavefront a stage, eight rows each.)
template <int NP> struct XRing {
  static constexpr int LOADS = (NP + 1) / 2, DEPTH = NP <= 4 ? 3 : 2;
  static constexpr unsigned BYTES = 64 * LOADS * 2 * TL_STRIDE;
  static_assert(DEPTH * BYTES <= TQ_X_BYTES, "the ring fits");
};

// The order in which a die's workgroups work its pairs.  The map lists tiles of experts with many rows first (the grouping kernel
// sorts them for this kernel) and `heavy` of them belong to experts of more than 128 rows: these wait for the matrix cores, the
// others for their weights.  Pairs of either kind are dealt to the dies in chunks, so that every die has as many of
// each height; a chunk is long enough for a tile's column blocks, which read the same activations, and an expert's row tiles, which
// read the same weights, to be worked on few dies.  A die works the heavy ones spread evenly among the others, so that at any
// time some workgroups multiply while the rest keep the memory busy, and a round of the lightest last, so that the last ones
// end soon after each other.  Where up to half of the places would have one more of these than the rest, that many go in halves (half the
// weight rows; nobody skips the products of the other half, which wait for nothing here): 68 pairs on 32 places of a die took three
// rounds of 24 us where the work is 2.1.
#define TQ_CHUNK 12
template <bool GATE_UP>
struct QueueList {
  static constexpr int ROWS = TL_ROWS(4), COLS = GATE_UP ? 128 : 256;
  struct Dealt {  // a run of pairs, the die's part of it
    unsigned whole, rest0, n;
    __device__ __forceinline__ Dealt(unsigned pairs, unsigned die) {
      whole = pairs / (8 * TQ_CHUNK) * TQ_CHUNK;
      const unsigned rest = pairs - 8 * whole;
      rest0 = 8 * whole + rest * die / 8;
      n = whole + 8 * whole + rest * (die + 1) / 8 - rest0;
    }
    __device__ __forceinline__ unsigned at(unsigned j, unsigned die) const {  // the j-th of the die's
      return j < whole ? (j / TQ_CHUNK * 8 + die) * TQ_CHUNK + j % TQ_CHUNK : rest0 + j - whole;
    }
  };
  const uint2* tiles;  // (first row, rows held and the rest, see ix_moe_dispatch)
  unsigned die;
  int heavy, n_col_blocks, each;  // each: row tiles of the second product
  Dealt first, many, few;
  unsigned many_seconds, halved, n;  // how many of `many` are the second product's, of the last pairs go in halves; the die's entries

  __device__ __forceinline__ QueueList(unsigned die_, const uint2* tiles_, int n_tiles, int heavy_, int n_col_blocks_, int width,
                                       const Second& second)
      : tiles(tiles_), die(die_), heavy(heavy_), n_col_blocks(n_col_blocks_), each((second.rows + ROWS - 1) / ROWS),
        // longer ones first: they then end with the others (88 of 88 stages beside some 600 of 22, of 256 places)
        first(second.width > width ? seconds(second) : 0u, die_),
        many((second.width > width ? 0u : seconds(second)) + static_cast<unsigned>(heavy_) * n_col_blocks_, die_),
        few(static_cast<unsigned>(n_tiles - heavy_) * n_col_blocks_, 7 - die_) {
    n = first.n + many.n + few.n;
    const unsigned over = n % (TQ_PLACES / 8);
    halved = over <= TQ_PLACES / 16 ? min(over, few.n) : 0u;
    n += halved;
    many_seconds = second.width > width ? 0u : seconds(second);
  }
  __device__ __forceinline__ static unsigned seconds(const Second& second) {
    return static_cast<unsigned>((second.rows + ROWS - 1) / ROWS) * static_cast<unsigned>((second.n_out + COLS - 1) / COLS);
  }

  // The i-th entry of the die, i < n: its tile (16 bits; the second product's: its row tile and TQ_SECOND), the half column block at which it
  // starts (15) and whether it ends there (1).
  __device__ __forceinline__ unsigned entry(unsigned i) const {
    bool of_second = false;
    unsigned at, half = 0, only = 0;
    if (i >= n - 2 * halved) {
      const unsigned j = i - (n - 2 * halved);
      at = few.at(few.n - halved + j / 2, 7 - die) + static_cast<unsigned>(heavy) * n_col_blocks;
      half = j & 1;
      only = 1u << 31;
    } else if (i < first.n) {
      of_second = true;
      at = first.at(i, die);
    } else {
      const unsigned q = i - first.n, last = min(few.n, static_cast<unsigned>(TQ_PLACES / 8)), mixed = many.n + few.n - last;
      const unsigned before = q < mixed ? q * many.n / mixed : many.n;
      if (q < mixed && (q + 1) * many.n / mixed > before) {
        at = many.at(before, die);
        of_second = at < many_seconds;
        at -= of_second ? 0u : many_seconds;
      } else {
        at = few.at(q - before, 7 - die) + static_cast<unsigned>(heavy) * n_col_blocks;
      }
    }
    if (of_second) return at % each | TQ_SECOND | at / each << 17;
    unsigned tile = at / n_col_blocks, col_block = at % n_col_blocks;
    // Row tiles of an expert that has several read the same weights: up to four of them one after the other for a column
    // block, so that all but the first find the weights in L2.
    const unsigned what = tiles[tile].y, start = tile - ((what >> 19) & 3u), together = ((what >> 21) & 3u) + 1;
    if (together > 1) {
      const unsigned in = at - start * n_col_blocks;
      tile = start + in % together;
      col_block = in / together;
    }
    return tile | (2 * col_block + half) << 16 | only;
  }
};

// What a workgroup works on, the same for all its lanes.
struct Work {
  const __bf16 *a, *w;  // w: the expert's
  const int32_t* rows;
  __bf16* out;
  int n_out, width, act, n0, end, row0, held, start;  // columns n0 to end; start: the number of the reduction at which stage 0 begins
  bool once;                                     // nobody else reads the weights

  __device__ __forceinline__ int place(int s) const {  // where stage s starts in a row
    const int k0 = s * TL_K + start;
    return k0 < width ? k0 : k0 - width;
  }
};

// (the same for all lanes, for the compiler too: a load's base is a pair of scalar registers)
template <typename T>
__device__ __forceinline__ T* uniform(T* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(v)), hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(v >> 32));
  return reinterpret_cast<T*>(lo | static_cast<uint64_t>(hi) << 32);
}

// The lane's rows of a Work, in bytes from its operand's start.
template <bool GATE_UP>
__device__ __forceinline__ void weight_rows(const Work& k, unsigned (&src)[4]) {
  const int r = 8 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + ((threadIdx.x & 63) >> 3);  // rows r, r + 64, r + 128, r + 192
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = GATE_UP ? (i < 2 ? 0 : k.n_out) + min(k.n0 + r + 64 * (i & 1), k.end - 1) : min(k.n0 + r + 64 * i, k.end - 1);
    src[i] = 2u * static_cast<unsigned>(row) * static_cast<unsigned>(k.width);
  }
}

// Weights of stage s to the buffer at `to`.
template <bool ONCE>
__device__ __forceinline__ void load_weights(__bf16* lds, const Work& k, const unsigned (&src)[4], unsigned to, int s, int piece, int wave) {
  const unsigned from = 2u * static_cast<unsigned>(k.place(s) + piece);
#pragma unroll
  for (int i = 0; i < 4; ++i) lds_load16<ONCE>(lds, to + 1024 * (wave + 8 * i), src[i] + from, uniform(k.w));
}
__device__ __forceinline__ void load_weights(__bf16* lds, const Work& k, const unsigned (&src)[4], unsigned to, int s, int piece, int wave) {
  if (k.once) load_weights<true>(lds, k, src, to, s, piece, wave);
  else load_weights<false>(lds, k, src, to, s, piece, wave);
}

// A Work's row numbers into LDS: the wavefront's 24 rows are lane >> 3 = i, lane & 7 of rows 8 (wave + 8 i) on.
__device__ __forceinline__ void load_row_numbers(__bf16* lds, const Work& k, int wave) {
  const int lane = threadIdx.x & 63;
  const int r = k.row0 + min(8 * (wave + 8 * (lane >> 3)) + (lane & 7), k.held - 1);
  lds_load4(lds, TQ_ROWS_AT + 256 * wave, 4u * static_cast<unsigned>(r), uniform(k.rows));
}
// ... which have arrived: the lane's activation rows, in bytes.  (Rows past the end repeat the last one.)
__device__ __forceinline__ void activation_rows(const __bf16* lds, const Work& k, unsigned (&src)[3], int wave) {
  const int sub = (threadIdx.x & 63) >> 3;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int row = k.rows ? reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(lds) + TQ_ROWS_AT + 256 * wave)[8 * i + sub]
                           : k.row0 + min(8 * (wave + 8 * i) + sub, k.held - 1);
    src[i] = 2u * static_cast<unsigned>(row) * static_cast<unsigned>(k.width);
  }
}

// The first stages' activations that the ring holds, and the third stage's weights; -> LOADS * (DEPTH - 1) + 4 loads behind stage 0's.
template <int NP>
__device__ __forceinline__ void load_activations(__bf16* lds, const Work& k, const unsigned (&src)[3], int piece, int wave) {
  using R = XRing<NP>;
#pragma unroll
  for (int s = 0; s < R::DEPTH; ++s) {
    const unsigned from = 2u * static_cast<unsigned>(k.place(s) + piece);
#pragma unroll
    for (int i = 0; i < R::LOADS; ++i) lds_load16<false>(lds, TQ_X_AT + s * R::BYTES + 1024 * (wave + 8 * i), src[i] + from, uniform(k.a));
  }
}
template <int NP> constexpr int behind_first() { return XRing<NP>::LOADS * (XRing<NP>::DEPTH - 1) + 4; }

__device__ __forceinline__ void load_start(__bf16* lds, const Work& k, const unsigned (&wsrc)[4], const unsigned (&xsrc)[3], unsigned third,
                                           int piece, int wave) {
  if (k.held <= 64) load_activations<2>(lds, k, xsrc, piece, wave);
  else if (k.held <= 128) load_activations<4>(lds, k, xsrc, piece, wave);
  else load_activations<6>(lds, k, xsrc, piece, wave);
  load_weights(lds, k, wsrc, third, 2, piece, wave);
}
// Until stage 0 of a Work has landed whose start was followed by LATER stores.
template <int LATER>
__device__ __forceinline__ void wait_start(const Work& k) {
  if (k.held <= 64) wait_loads<behind_first<2>() + LATER>();
  else if (k.held <= 128) wait_loads<behind_first<4>() + LATER>();
  else wait_loads<behind_first<6>() + LATER>();
}

// What goes from pair to pair.
struct Run {
  Work k;
  unsigned wsrc[4], xsrc[3];
  unsigned wbuf;  // where stage 0's weights lie
};

// One pair, whose stage 0 lies in LDS and whose next ones are on their way; the next pair is started.  false: there is none.
// NP: pairs of sixteens of activation rows the tile holds, one of each a wavefront.  (Wavefronts, products and reads as in tiled_body.)
template <bool GATE_UP, int NP, bool ONCE, typename Take, typename Fetch, typename Fetched>
__device__ __forceinline__ bool queue_body(Run& run, __bf16* lds, float glu_limit, Take take, Fetch fetch, Fetched fetched) {
  using R = XRing<NP>;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 15, g = lane >> 4, wi = wave & 3, xi = wave >> 2;
  const int piece = 8 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4)));
  constexpr int HALF = 128;
  const Work& k = run.k;
  const __bf16 *const ka = uniform(k.a), *const kw = uniform(k.w);
  const int stages = k.width / TL_K;

  f32x4 acc[4][NP];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int t = 0; t < NP; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int xat[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) xat[kk] = tl_at(m, 4 * kk + g);
  const __bf16* const ws = lds + (GATE_UP ? 32 : 64) * wi * TL_STRIDE;
  const __bf16* const xs = lds + TQ_X_AT / 2 + 16 * xi * TL_STRIDE;
  struct Half { bf16x8 w[4], x[NP]; };
  Half h0, h1;
  unsigned wbuf = run.wbuf, xbuf = 0;
  auto read = [&](Half& h, int i, int kk) {  // the i-th of a half's NP + 4 pieces
    if (i < 4) {
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
  for (int i = 0; i < NP + 4; ++i) read(h0, i, 0);

  Work next;
  unsigned nsrc[4];
  bool more = false;
  // Stage s, the operands of its first half in registers; LEFT: at least so many stages follow.
  constexpr int READS = NP > 1 ? (NP + 4 + NP - 2) / (NP - 1) : 5, LOADS = (4 + R::LOADS + NP - 1) / NP;
  auto stage = [&](auto left, int s) {
    constexpr int LEFT = decltype(left)::value;
#pragma unroll
    for (int t = 0; t < NP; ++t) {
      products(h0, t);
#pragma unroll
      for (int i = READS * t; i < READS * (t + 1); ++i) read(h1, i, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // Stage s + 1 must have landed.  After its last load there were issued (an iteration issues activations first) the weights of
    // stages up to s + TQ_W - 1 and the activations of stages up to s + DEPTH - 1, as far as there are so many.
    if constexpr (LEFT > 1) wait_loads<4 + R::LOADS * (R::DEPTH - 2)>();
    else wait_loads<0>();
    if constexpr (LEFT == 1) fetched();
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const unsigned wfree = wbuf, xfree = xbuf;  // nobody reads stage s any more
    wbuf = wbuf + TQ_WT == TQ_W * TQ_WT ? 0 : wbuf + TQ_WT;
    xbuf = xbuf + R::BYTES == R::DEPTH * R::BYTES ? 0 : xbuf + R::BYTES;
    if constexpr (LEFT == 1) {
      more = take(next);
      if (more) {
        if (next.rows) load_row_numbers(lds, next, wave);
        weight_rows<GATE_UP>(next, nsrc);
        load_weights(lds, next, nsrc, wbuf + TQ_WT == TQ_W * TQ_WT ? 0 : wbuf + TQ_WT, 0, piece, wave);  // (of stage s - 1)
        load_weights(lds, next, nsrc, wfree, 1, piece, wave);
      }
    }
    const unsigned from_x = LEFT >= R::DEPTH ? 2u * static_cast<unsigned>(k.place(s + R::DEPTH) + piece) : 0u;
    const unsigned from_w = LEFT >= TQ_W ? 2u * static_cast<unsigned>(k.place(s + TQ_W) + piece) : 0u;
#pragma unroll
    for (int t = 0; t < NP; ++t) {
      products(h1, t);
#pragma unroll
      for (int i = READS * t; i < READS * (t + 1); ++i) read(h0, i, 0);
#pragma unroll
      for (int i = LOADS * t; i < LOADS * (t + 1); ++i) {
        if (i < R::LOADS) {
          if constexpr (LEFT >= R::DEPTH) lds_load16<false>(lds, TQ_X_AT + xfree + 1024 * (wave + 8 * i), run.xsrc[i] + from_x, ka);
        } else if (i < R::LOADS + 4) {
          if constexpr (LEFT >= TQ_W) lds_load16<ONCE>(lds, wfree + 1024 * (wave + 8 * (i - R::LOADS)), run.wsrc[i - R::LOADS] + from_w, kw);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int s = 0; s < stages - 4; ++s) stage(std::integral_constant<int, 3>{}, s);
  fetch();
  stage(std::integral_constant<int, 3>{}, stages - 4);
  stage(std::integral_constant<int, 2>{}, stages - 3);
  stage(std::integral_constant<int, 1>{}, stages - 2);
  // the last one
#pragma unroll
  for (int t = 0; t < NP; ++t) {
    products(h0, t);
#pragma unroll
    for (int i = READS * t; i < READS * (t + 1); ++i) read(h1, i, 1);
    __builtin_amdgcn_sched_barrier(0);
  }
  lds_barrier();  // nobody reads the rings any more; the next pair's first two stages of weights are on their way to two of three buffers
  __builtin_amdgcn_sched_barrier(0);
  unsigned nx[3];
  if (more) {
    if (next.rows) wait_loads<8>();  // (the row numbers; the weights after them)
    activation_rows(lds, next, nx, wave);
    load_start(lds, next, nsrc, nx, wbuf, piece, wave);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < NP; ++t) products(h1, t);

  // The lane holds weight rows (block) + 4 g + i of activation row row0 + 16 (2 t + xi) + m.  Two lanes that differ by 16 exchange
  // their fours of two blocks, so that each has eight columns of one: a store is 16 bytes a lane, 64 of a row.  Rows past the
  // end hold the last one's results and go there, too, so that every wavefront has the same number of stores.
  const bool partial = k.n0 + (GATE_UP ? HALF : 2 * HALF) > k.end;
#pragma unroll
  for (int t = 0; t < NP; ++t) {
    const int64_t row = k.row0 + min(16 * (2 * t + xi) + m, k.held - 1);
#pragma unroll
    for (int pair = 0; pair < (GATE_UP ? 1 : 2); ++pair) {
      unsigned two[2][2];  // block, pair of columns
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int j = 2 * pair + b;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = acc[j][t][i];
          if (GATE_UP) v[i] = ix_glu<true>(v[i], acc[GATE_UP ? j + 2 : j][t][i], glu_limit);
          else if (k.act) v[i] = v[i] > 0.f ? v[i] * v[i] : 0.f;  // the square of relu
        }
        two[b][0] = ix_f32x2_to_bf16x2(v[0], v[1]);
        two[b][1] = ix_f32x2_to_bf16x2(v[2], v[3]);
      }
      const auto lo = __builtin_amdgcn_permlane16_swap(two[0][0], two[1][0], false, false);
      const auto hi = __builtin_amdgcn_permlane16_swap(two[0][1], two[1][1], false, false);
      const int c = k.n0 + (GATE_UP ? 32 : 64) * wi + 16 * (2 * pair + (g & 1)) + 8 * (g >> 1);
      if (!partial || c < k.end)
        *reinterpret_cast<uint4*>(k.out + row * k.n_out + c) = make_uint4(lo[0], hi[0], lo[1], hi[1]);
    }
  }
  if (!more) return false;
  if (partial) wait_start<0>(next);  // (some wavefronts have fewer stores)
  else wait_start<(GATE_UP ? 1 : 2) * NP>(next);
  lds_barrier();
  run.k = next;
  run.wbuf = wbuf + TQ_WT == TQ_W * TQ_WT ? 0 : wbuf + TQ_WT;
#pragma unroll
  for (int i = 0; i < 4; ++i) run.wsrc[i] = nsrc[i];
#pragma unroll
  for (int i = 0; i < 3; ++i) run.xsrc[i] = nx[i];
  return true;
}

// queue: a counter a die, 0 before the first launch with it, and the number of tiles of experts with more than 128 rows.
// tiles: the map's, most rows first (see ix_moe_dispatch); places for max_tiles of them.
template <bool GATE_UP>
__global__ void __launch_bounds__(TQ_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
moe_grouped_queue_kernel(const __bf16* a, const __bf16* w, __bf16* out, const int32_t* rows, const uint2* __restrict__ tiles,
                         const int32_t* __restrict__ tile_info, int max_tiles, int32_t* queue, int n_out, int width, int n_col_blocks,
                         int act, float glu_limit, Second second) {
  __shared__ __attribute__((aligned(1024))) __bf16 lds[TQ_LDS / 2];
  const unsigned die = blockIdx.x & 7;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int piece = 8 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4)));
  int* const next_at = reinterpret_cast<int*>(reinterpret_cast<char*>(lds) + TQ_NEXT_AT);
  uint2* const held = reinterpret_cast<uint2*>(reinterpret_cast<char*>(lds) + TQ_TILES_AT);
  unsigned* const items = reinterpret_cast<unsigned*>(reinterpret_cast<char*>(lds) + TQ_LIST_AT);
  // (places past the last tile hold anything, and nobody looks there)
  for (int i = tid; i < max_tiles; i += TQ_THREADS) held[i] = tiles[i];
  const QueueList<GATE_UP> list(die, held, tile_info[0], queue[8], n_col_blocks, width, second);
  const unsigned n = min(list.n, static_cast<unsigned>(TQ_LIST));  // (no more: the entry point has counted)
  if ((blockIdx.x >> 3) >= n) return;
  auto work = [&](unsigned item) {
    item = __builtin_amdgcn_readfirstlane(item);
    const bool of_second = item & TQ_SECOND;
    const unsigned tile = item & (TQ_SECOND - 1);
    const uint2 d = held[of_second ? 0 : tile];
    const unsigned what = __builtin_amdgcn_readfirstlane(d.y), e = of_second ? 0u : (what >> 8) & 2047u;
    Work k;
    k.a = of_second ? second.a : a;
    k.rows = of_second ? nullptr : rows;
    k.out = of_second ? second.out : out;
    k.n_out = of_second ? second.n_out : n_out;
    k.width = of_second ? second.width : width;
    k.act = of_second ? 0 : act;
    k.w = of_second ? second.w : w + static_cast<int64_t>(e) * (GATE_UP ? 2 * static_cast<int64_t>(n_out) : n_out) * width;
    k.n0 = static_cast<int>(item >> 16 & 32767u) * (GATE_UP ? 64 : 128);
    k.end = min(k.n0 + (GATE_UP ? 128 : 256) / (item >> 31 ? 2 : 1), k.n_out);
    k.row0 = of_second ? TL_ROWS(4) * static_cast<int>(tile) : static_cast<int>(__builtin_amdgcn_readfirstlane(d.x));
    k.held = of_second ? min(TL_ROWS(4), second.rows - k.row0) : static_cast<int>(what & 255u);
    k.once = !of_second && (what >> 23 & 1) && (reinterpret_cast<uintptr_t>(w) & 127) == 0;  // (whole lines)
    // (experts start at different stages, see tiled_body)
    k.start = k.width % 512 == 0 ? static_cast<int>((e * 3u) % static_cast<unsigned>(k.width / TL_K)) * TL_K : 0;
    return k;
  };
  int got = 0;
  auto fetch = [&]() {
    if (tid == 0) got = __hip_atomic_fetch_add(queue + die, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  // A die's workgroups ask once a pair, n times in all: whoever asks last leaves the counter as the next launch with it needs it.
  auto fetched = [&]() {
    if (tid == 0) {
      const int before = got & (TQ_USED - 1);
      *next_at = TQ_PLACES / 8 + before;
      if (before == static_cast<int>(n) - 1) __hip_atomic_store(queue + die, TQ_USED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  auto take = [&](Work& next) {
    const unsigned i = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(*next_at));
    if (i < n) next = work(items[i]);
    return i < n;
  };
  __syncthreads();
  Run run;
  run.k = work(list.entry(blockIdx.x >> 3));
  run.wbuf = 0;
  weight_rows<GATE_UP>(run.k, run.wsrc);
  if (run.k.rows) load_row_numbers(lds, run.k, wave);
  load_weights(lds, run.k, run.wsrc, 0, 0, piece, wave);
  load_weights(lds, run.k, run.wsrc, TQ_WT, 1, piece, wave);
  if (run.k.rows) wait_loads<8>();
  activation_rows(lds, run.k, run.xsrc, wave);
  load_start(lds, run.k, run.wsrc, run.xsrc, 2 * TQ_WT, piece, wave);
  for (unsigned i = tid; i < n; i += TQ_THREADS) items[i] = list.entry(i);  // while these are on their way
  wait_start<0>(run.k);
  lds_barrier();
  for (bool more = true; more;) {
#define BODY(NP)                                                                                                            \
  more = run.k.once ? queue_body<GATE_UP, NP, true>(run, lds, glu_limit, take, fetch, fetched)                              \
                    : queue_body<GATE_UP, NP, false>(run, lds, glu_limit, take, fetch, fetched)
    switch ((run.k.held + 31) >> 5) {  // pairs of sixteens of rows this tile holds
      case 1: BODY(1); break;
      case 2: BODY(2); break;
      case 3: BODY(3); break;
      case 4: BODY(4); break;
      case 5: BODY(5); break;
      default: BODY(6); break;
    }
#undef BODY
  }
}

// Whether the staying workgroups take a product's operands: whole stages, at least four of them, and results stored 16 bytes at a time.
static bool whole(int64_t n_out, int64_t width, const void* a, const void* w, const void* out) {
  return width % TL_K == 0 && width >= 4 * TL_K && n_out % 8 == 0 &&
         ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
}

// As ix_moe_grouped_tiled's wide form (which has checked sizes); -> 2, and nothing queued, where it has to do the product.
int ix_moe_grouped_queue(const void* a, const void* w, void* out, const int32_t* rows, const int32_t* tile_info, const void* tiles,
                         int32_t* queue, int max_tiles, int64_t n_out, int64_t width, int gate_up, float glu_limit, const void* a2, const void* w2,
                         void* out2, int64_t rows2, int64_t n_out2, int64_t width2, hipStream_t stream) {
  const int64_t cols = gate_up == 1 ? 128 : 256, blocks = (n_out + cols - 1) / cols, blocks2 = rows2 ? (n_out2 + cols - 1) / cols : 0;
  const int64_t pairs = blocks * max_tiles + blocks2 * ((rows2 + TL_ROWS(4) - 1) / TL_ROWS(4));
  if (max_tiles > TQ_TILES || pairs / 8 + 3 + TQ_PLACES / 16 > TQ_LIST || rows2 >= int64_t(TQ_SECOND) * TL_ROWS(4) || !whole(n_out, width, a, w, out)) return 2;
  if (rows2 && !whole(n_out2, width2, a2, w2, out2)) return 2;
  const Second second{(const __bf16*)a2, (const __bf16*)w2, (__bf16*)out2, (int)rows2, (int)n_out2, (int)width2};
#define LAUNCH(GU)                                                                                                             \
  hipLaunchKernelGGL((moe_grouped_queue_kernel<GU>), dim3(TQ_PLACES), dim3(TQ_THREADS), 0, stream, (const __bf16*)a,            \
                     (const __bf16*)w, (__bf16*)out, rows, (const uint2*)tiles, tile_info, max_tiles, queue, (int)n_out, (int)width, (int)blocks,  \
                      gate_up == 2 ? 1 : 0, glu_limit, second)
  if (gate_up == 1) LAUNCH(true);
  else LAUNCH(false);
#undef LAUNCH
  return ix_check_launch("ix_moe_grouped_tiled");
}
