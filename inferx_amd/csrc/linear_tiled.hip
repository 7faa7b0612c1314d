// Dense products out[rows, n_out] = x[rows, width] . w[n_out, width]^T for a few dozen to some hundred rows, bfloat16 operands,
// 32-bit accumulation, out bfloat16 or float32: more rows than linear_skinny's few, and fewer tiles than the vendor's library
// needs to fill the chip.
//
// A workgroup owns a tile of weight rows x activation rows; stages of 64 of the reduction go through a ring of LDS
// buffers that the loads fill by themselves, as in moe_tiled.hip (halves of 32, one barrier a stage, LDS rows with their
// 16-byte pieces permuted).  The product is formed transposed (A = weight rows), WI x XI wavefronts own WB sixteens of weight rows and
// XB of activation rows each.
//
// What bounds it: what a compute unit takes from L2.  With one tile a compute unit every form from 32 x 32 to 128 x 192 takes
// 5 us and the bytes of its stages at 53 to 61 GB/s; two stages of 64 a barrier change nothing.  So the tile with the fewest rows
// of both kinds (its bytes a stage) whose number fits the chip's 256 compute units is the fastest, and the library, which
// takes 64 x 64 and more for few rows, is slower as long as there is one.  Weights from memory, us, against the library: 64 x 2,048
// x 6,144 12.6 (18.9), 64 x 2,048 x 2,048 11.0 (15.8), 340 x 2,048 x 6,144 23.8 (31.9), 512 x 3,584 x 4,608 39.5 (41.6),
// 850 x 2,048 x 6,144 29.7 (34.7), 2,048 x 2,048 x 2,048 26.5 (29.0).
// With up to 64 rows and so many weights that memory bounds the product, two workgroups of 128 x 64 share a compute unit: 64 x 2,048 x
// 151,936 to float32 125 us (204; the weights alone take 97).
#include <type_traits>

#include "lds_loads.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define LT_K 64        // numbers of the reduction a stage
#define LT_STRIDE 64   // numbers of an LDS row
#define LT_UNITS 256   // compute units
__device__ __forceinline__ int lt_at(int row, int piece) { return row * LT_STRIDE + ((piece ^ ((row >> 1) & 7)) << 3); }

template <int WI_, int XI_, int WB_, int XB_, int RING_> struct LinearTile {
  static constexpr int WI = WI_, XI = XI_, WB = WB_, XB = XB_, RING = RING_, WAVES = WI * XI;
  static constexpr int W = 16 * WB * WI, X = 16 * XB * XI;  // weight and activation rows
  static constexpr int BYTES = RING * (W + X) * 2 * LT_STRIDE;
  static_assert(BYTES <= 163840 && X * (W + 8) * 2 <= BYTES, "the ring fits LDS, and the result's tile the ring");
  static_assert(WAVES % 2 == 0 && W % (8 * WAVES) == 0 && X % (8 * WAVES) == 0, "whole loads for every wavefront");
};

// NT: the weights are read by one row tile only and their rows are whole lines: past the caches.  (Rows that share lines would bring those
// from memory for each of them: tiles of 128 x 64 with a reduction that is not made of whole lines 0.94 of the time through the caches.)
template <typename T, bool NT, bool F32>
__global__ void __launch_bounds__(64 * T::WAVES) __attribute__((amdgpu_waves_per_eu(1, 2)))
linear_tiled_kernel(const __bf16* x, const __bf16* w, void* out, int rows, int n_out, int width, int row_tiles) {
  constexpr int WB = T::WB, XB = T::XB, RING = T::RING, WAVES = T::WAVES;
  constexpr int NPX = T::X / 8 / WAVES, PER = T::W / 8 / WAVES + NPX;  // loads of a wavefront a stage, eight rows each
  constexpr unsigned WT = T::W * 2 * LT_STRIDE, XT = T::X * 2 * LT_STRIDE;  // bytes of a stage
  __shared__ __attribute__((aligned(1024))) __bf16 lds[T::BYTES / 2];
  // The row tiles of a block of weight rows go to one die one after the other, as they read the same weights: the pairs,
  // block by block, are cut into eight runs, one a die (workgroup i goes to die i % 8).
  const unsigned die = blockIdx.x & 7, each = gridDim.x >> 3, more = gridDim.x & 7;  // the first `more` dies have one pair more
  const unsigned pair = die * each + min(die, more) + (blockIdx.x >> 3);
  const int block = static_cast<int>(pair / row_tiles), n0 = block * T::W, row0 = static_cast<int>(pair % row_tiles) * T::X;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4, wi = wave % T::WI, xi = wave / T::WI;

  // where this lane's rows start, in bytes: a wavefront brings rows 8 (wave + WAVES i) to + 7 (past the end the last one again)
  const __bf16* const w_block = w + static_cast<int64_t>(n0) * width;
  unsigned src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int r = 8 * (wave + WAVES * (i < NPX ? i : i - NPX)) + (lane >> 3);
    src[i] = 2u * static_cast<unsigned>(i < NPX ? min(row0 + r, rows - 1) : min(r, n_out - 1 - n0)) * static_cast<unsigned>(width);
  }
  // what belongs at piece lane & 7 of the lane's rows (the number of a wavefront's eights is as odd or even as its own)
  const int piece = 8 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4)));
  // Blocks start the reduction at different stages and wrap round (see moe_tiled.hip): rows of a multiple of 1,024 bytes
  // would all ask the same memory channels at once.
  const int stages = (width + LT_K - 1) / LT_K, kspan = stages * LT_K;
  const int rot = width % 512 == 0 ? static_cast<int>((static_cast<unsigned>(block) * 3u) % static_cast<unsigned>(stages)) * LT_K : 0;
  auto place = [&](int s) {  // where stage s starts in a row (past the end: the last stage again)
    const int k0 = min(s * LT_K, kspan - LT_K);
    return k0 + rot < kspan ? k0 + rot : k0 + rot - kspan;
  };
  // (a piece that does not exist, where the width is no multiple of 64, is the row's last one; zeros take its place)
  auto at = [&](int s) { return 2u * static_cast<unsigned>(min(place(s) + piece, width - 8)); };
  auto load = [&](int buf, int i, unsigned from) {  // the i-th of a stage's loads
    if (i < NPX) lds_load16<false>(lds, RING * WT + buf * XT + 1024 * (wave + WAVES * i), src[i] + from, x);
    else if (i < PER) lds_load16<NT>(lds, buf * WT + 1024 * (wave + WAVES * (i - NPX)), src[i] + from, w_block);
  };

  f32x4 acc[WB][XB];
#pragma unroll
  for (int j = 0; j < WB; ++j)
#pragma unroll
    for (int t = 0; t < XB; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int xat[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) xat[kk] = lt_at(m, 4 * kk + g);
  const __bf16* const ws = lds + 16 * WB * wi * LT_STRIDE;
  const __bf16* const xs = lds + RING * WT / 2 + 16 * XB * xi * LT_STRIDE;
  struct Half { bf16x8 w[WB], x[XB]; };
  Half h0, h1;
  auto read = [&](Half& h, int i, int buf, int kk) {  // the i-th of a half's WB + XB pieces
    if (i < WB) h.w[i] = *reinterpret_cast<const bf16x8*>(ws + buf * (WT / 2) + xat[kk] + 16 * i * LT_STRIDE);
    else if (i < WB + XB) h.x[i - WB] = *reinterpret_cast<const bf16x8*>(xs + buf * (XT / 2) + xat[kk] + 16 * (i - WB) * LT_STRIDE);
  };
  auto products = [&](const Half& h, int t) {
#pragma unroll
    for (int j = 0; j < WB; ++j) acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h.w[j], h.x[t], acc[j][t], 0, 0, 0);
  };

#pragma unroll
  for (int s = 0; s < RING; ++s)
#pragma unroll
    for (int i = 0; i < PER; ++i) load(s, i, at(s));
  wait_loads<PER * (RING - 1)>();
  lds_barrier();
  int buf = 0;
#pragma unroll
  for (int i = 0; i < WB + XB; ++i) read(h0, i, buf, 0);
  // Stage s, the operands of its first half in registers; LEFT: at least so many stages follow.  Reads and loads go between
  // the products, as many a step as leave the last ones time to arrive.
  constexpr int READS = XB > 1 ? (WB + XB + XB - 2) / (XB - 1) : WB + XB, LOADS = (PER + XB - 1) / XB;
  auto stage = [&](auto left, int s) {
    constexpr int LEFT = decltype(left)::value;
#pragma unroll
    for (int t = 0; t < XB; ++t) {
      if constexpr (LEFT > 0) products(h0, t);
#pragma unroll
      for (int i = READS * t; i < READS * (t + 1); ++i) read(h1, i, buf, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LEFT == 0) {
      if (width & (LT_K - 1)) {  // the last stage is not whole
        const bf16x8 zero = {(__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f,
                             (__bf16)0.f, (__bf16)0.f, (__bf16)0.f, (__bf16)0.f};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
          if (place(s) + 32 * kk + 8 * g >= width) {
            Half& h = kk ? h1 : h0;
#pragma unroll
            for (int j = 0; j < WB; ++j) h.w[j] = zero;
#pragma unroll
            for (int t = 0; t < XB; ++t) h.x[t] = zero;
          }
      }
#pragma unroll
      for (int t = 0; t < XB; ++t) products(h0, t);
#pragma unroll
      for (int t = 0; t < XB; ++t) products(h1, t);
    } else {
      wait_loads<PER * (RING - 2 < LEFT - 1 ? RING - 2 : LEFT - 1)>();  // stage s + 1 has landed
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
      const int free = buf;  // nobody reads stage s any more
      buf = buf + 1 == RING ? 0 : buf + 1;
      const unsigned from = LEFT >= RING ? at(s + RING) : 0u;
#pragma unroll
      for (int t = 0; t < XB; ++t) {
        products(h1, t);
#pragma unroll
        for (int i = READS * t; i < READS * (t + 1); ++i) read(h0, i, buf, 0);
        if constexpr (LEFT >= RING)
#pragma unroll
          for (int i = LOADS * t; i < LOADS * (t + 1); ++i) load(free, i, from);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
#define LT_STAGE(LEFT, S) stage(std::integral_constant<int, (LEFT)>{}, (S))
  int s = 0;
  for (; s < stages - RING; ++s) LT_STAGE(RING, s);
  // the last ones, for which everything has been asked for: once the first has let the others go on arriving, all have
  if (s < stages - 1 && stages - 1 - s >= RING - 1) {
    LT_STAGE(RING - 1, s);
    ++s;
  }
  for (; s < stages - 1; ++s) LT_STAGE(1, s);
  LT_STAGE(0, stages - 1);
#undef LT_STAGE
  wait_loads<0>();  // (with fewer stages than the ring holds, the last one again)

  // lane holds weight rows n0 + 16 (WB wi + j) + 4 g + i of activation row row0 + 16 (XB xi + t) + m
  if constexpr (!F32) {
    if (((n_out & 7) | static_cast<int>(reinterpret_cast<uintptr_t>(out) & 15)) == 0) {
      // The tile goes through LDS, so that a store is 16 bytes a lane and whole lines.
      constexpr int OUT_STRIDE = T::W + 8, LANES = T::W / 8, AT_ONCE = 64 * WAVES / LANES;  // lanes of a row; rows stored at once
      __syncthreads();
#pragma unroll
      for (int t = 0; t < XB; ++t)
#pragma unroll
        for (int j = 0; j < WB; ++j)
          *reinterpret_cast<bf16x4*>(lds + (16 * (XB * xi + t) + m) * OUT_STRIDE + 16 * (WB * wi + j) + 4 * g) =
              bf16x4{(__bf16)acc[j][t][0], (__bf16)acc[j][t][1], (__bf16)acc[j][t][2], (__bf16)acc[j][t][3]};
      __syncthreads();
      const int c = 8 * (tid % LANES);
      if (n0 + c < n_out && tid < AT_ONCE * LANES)
        for (int r = tid / LANES; r < min(T::X, rows - row0); r += AT_ONCE)
          *reinterpret_cast<bf16x8*>(static_cast<__bf16*>(out) + static_cast<int64_t>(row0 + r) * n_out + n0 + c) =
              *reinterpret_cast<const bf16x8*>(lds + r * OUT_STRIDE + c);
      return;
    }
  }
  const bool vec = F32 && (n_out & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
  for (int t = 0; t < XB; ++t) {
    const int r = row0 + 16 * (XB * xi + t) + m;
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < WB; ++j) {
      const int nb = n0 + 16 * (WB * wi + j) + 4 * g;
      const int64_t to = static_cast<int64_t>(r) * n_out + nb;
      if (vec && nb + 4 <= n_out) {
        *reinterpret_cast<f32x4*>(static_cast<float*>(out) + to) = acc[j][t];
        continue;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (nb + i < n_out) {
          if constexpr (F32) static_cast<float*>(out)[to + i] = acc[j][t][i];
          else static_cast<__bf16*>(out)[to + i] = (__bf16)acc[j][t][i];
        }
    }
  }
}

namespace {

template <typename T>
int64_t tiles_of(int64_t rows, int64_t n_out) { return ((rows + T::X - 1) / T::X) * ((n_out + T::W - 1) / T::W); }

template <typename T>
int linear_tiled(const void* x, const void* w, void* out, int64_t rows, int64_t n_out, int64_t width, int out_f32,
                 hipStream_t stream) {
  const int64_t row_tiles = (rows + T::X - 1) / T::X, tiles = tiles_of<T>(rows, n_out);
  IX_REQUIRE(tiles < (int64_t(1) << 31), "too many workgroups for one launch");
#define LAUNCH(NT, F)                                                                                                    \
  hipLaunchKernelGGL((linear_tiled_kernel<T, NT, F>), dim3(static_cast<unsigned>(tiles)), dim3(64 * T::WAVES), 0, stream, \
                     (const __bf16*)x, (const __bf16*)w, out, (int)rows, (int)n_out, (int)width, (int)row_tiles)
  if (row_tiles == 1 && width % LT_K == 0 && (reinterpret_cast<uintptr_t>(w) & 127) == 0) {  // (whole lines)
    if (out_f32) LAUNCH(true, true);
    else LAUNCH(true, false);
  } else {
    if (out_f32) LAUNCH(false, true);
    else LAUNCH(false, false);
  }
#undef LAUNCH
  return ix_check_launch("ix_linear_tiled");
}

// by the rows of both kinds that a tile has
using Tile0 = LinearTile<2, 2, 1, 1, 10>;  // 32 x 32
using Tile1 = LinearTile<2, 2, 1, 2, 6>;   // 32 x 64
using Tile2 = LinearTile<2, 2, 2, 2, 5>;   // 64 x 64
using Tile3 = LinearTile<2, 2, 2, 3, 6>;   // 64 x 96
using Tile4 = LinearTile<2, 2, 2, 4, 6>;   // 64 x 128
using Tile5 = LinearTile<2, 2, 3, 4, 5>;   // 96 x 128
using Tile6 = LinearTile<4, 2, 2, 4, 5>;   // 128 x 128
using Tile7 = LinearTile<2, 4, 4, 3, 4>;   // 128 x 192
using TileN = LinearTile<2, 2, 4, 2, 3>;   // 128 x 64, two workgroups a compute unit

}  // namespace

// The tile for a product, or -1: the one with the fewest rows of both kinds whose number fits the compute units.  Up to 64 rows of
// what does not fit go in tiles of 128 x 64 (a vocabulary's weights: 33 rows of 151,936 x 2,048 116 us, 197 through the library, 64
// rows 125 against 199).  Over 3,460 products of 17 to 3,000 rows the tiles take 0.71 of the library's time (geometric mean) where these
// lines leave it to them, and 1.02 where they do not:
//   Up to 128 tiles of 32 x 32 with a long reduction: the library cuts it (5,120 to 22,000: 1.05; 663 x 15,872 x 24 38 against 16
// us, 66 x 8,704 x 192 21.7 against 10.7, 37 x 7,680 x 192 18.6 against 9.9; up to 5,120 0.7, of more tiles 0.8).
//   Results of no whole fours a row, which are stored one by one: from 64 x 96 on 0.99 (780 x 480 x 6,355 21.8 against 16.9).
//   64 x 128 with more than 4,096 of reduction where a fifth of the units have none (180 of them at 640 x 5,632 x 2,304 33.1 against 29.9;
// 818 x 5,632 x 2,048, 224 tiles, 31.0 against 32.4), 128 x 128 and 128 x 192 from 2,048 of reduction on (850 x 3,584 x 3,584 39.8 against
// 38.1; 682 x 3,584 x 4,608, 216 tiles, 37.4 against 43.5).  96 x 128 and larger also where many stages follow, which are long enough for the
// library to be ahead (1,400 x 5,632 x 2,048 55.7 against 52.1), or up to three (3,000 x 64 x 700 11.3 against 10.3; 1,500 x 512 x
// 2,048 11.4 against 14.6).
static int tile_for(int64_t rows, int64_t n_out, int64_t width) {
  const int64_t tiles[8] = {tiles_of<Tile0>(rows, n_out), tiles_of<Tile1>(rows, n_out), tiles_of<Tile2>(rows, n_out),
                            tiles_of<Tile3>(rows, n_out), tiles_of<Tile4>(rows, n_out), tiles_of<Tile5>(rows, n_out),
                            tiles_of<Tile6>(rows, n_out), tiles_of<Tile7>(rows, n_out)};
  int tile = 0;
  while (tile < 8 && tiles[tile] > LT_UNITS) ++tile;
  if (tile == 0 && width > 5120 && 2 * tiles[0] <= LT_UNITS) return -1;
  if (tile > 4 && rows <= TileN::X) return 8;
  if (tile > 2 && n_out % 4 != 0) return -1;
  if (tile == 8 || (tile > 4 && (width > 4096 || width < 256))) return -1;
  if (5 * tiles[tile] < 4 * LT_UNITS && ((tile == 4 && width > 4096) || (tile > 5 && width > 2048))) return -1;
  return tile;
}

// (a lane's place in its block of weights, and in the activations, is counted in 32 bits of bytes)
static bool small_enough(int64_t rows, int64_t n_out, int64_t width) {
  return rows * width < (int64_t(1) << 31) && 256 * width < (int64_t(1) << 31) && n_out < (int64_t(1) << 31) - 512;
}

// The rule's tile for a product, 0 to 8, or -1.
extern "C" int ix_linear_tiled_tile(int64_t rows, int64_t n_out, int64_t width) {
  if (rows <= 0 || n_out <= 0 || width <= 0 || width % 8 != 0 || !small_enough(rows, n_out, width)) return -1;
  return tile_for(rows, n_out, width);
}

// Operands on 16-byte boundaries.  tile: 0 to 8 that one, -1 the rule chooses; then 2 is returned, and nothing queued, where it has
// no tile for the product.
extern "C" int ix_linear_tiled(const void* x, const void* w, void* out, int64_t rows, int64_t n_out, int64_t width,
                               int out_f32, int tile, hipStream_t stream) {
  IX_REQUIRE(rows > 0 && n_out > 0 && width > 0, "sizes must be positive");
  IX_REQUIRE(width % 8 == 0, "the reduction width must be a multiple of 8");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) == 0, "operands must lie on 16-byte boundaries");
  if (tile < 0) {
    tile = ix_linear_tiled_tile(rows, n_out, width);
    if (tile < 0) return 2;
  }
  IX_REQUIRE(small_enough(rows, n_out, width), "sizes too large");
  switch (tile) {
    case 0: return linear_tiled<Tile0>(x, w, out, rows, n_out, width, out_f32, stream);
    case 1: return linear_tiled<Tile1>(x, w, out, rows, n_out, width, out_f32, stream);
    case 2: return linear_tiled<Tile2>(x, w, out, rows, n_out, width, out_f32, stream);
    case 3: return linear_tiled<Tile3>(x, w, out, rows, n_out, width, out_f32, stream);
    case 4: return linear_tiled<Tile4>(x, w, out, rows, n_out, width, out_f32, stream);
    case 5: return linear_tiled<Tile5>(x, w, out, rows, n_out, width, out_f32, stream);
    case 6: return linear_tiled<Tile6>(x, w, out, rows, n_out, width, out_f32, stream);
    case 7: return linear_tiled<Tile7>(x, w, out, rows, n_out, width, out_f32, stream);
    case 8: return linear_tiled<TileN>(x, w, out, rows, n_out, width, out_f32, stream);
    default: IX_REQUIRE(false, "no such tile"); return 1;
  }
}
