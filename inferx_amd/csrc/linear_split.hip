// Dense float32 products out[rows, n_out] = x[rows, width] . w[n_out, width]^T for prompt portions, on the bfloat16 matrix cores
// (see split_f32.h).
//
// The activations are split beforehand (`ix_split_rows`, 5 us): a row's every 32 numbers are 32 of each part, side by side.  The weights
// stay float32 and are split in registers, sixteen numbers of the reduction ahead of the products, so that the vector unit works
// beside the matrix cores; at most one other wavefront of the workgroup splits the same.  (With both operands split in the kernel, 64 x 64 of
// a wavefront, the eleven instructions for two numbers took longer than the products: 511 rows of 2,048 x 11,264 142 us, now 119.)
//
// A workgroup owns a tile of weight rows x activation rows, a wavefront 32 weight rows x one or two blocks of 32 activation rows.  Stages
// of 32 of the reduction go through a ring of LDS buffers that the loads fill by themselves.  The 16-byte pieces of LDS rows are
// permuted, so that what a quarter of a wavefront reads falls on different banks.  Tiles of 64 x 64 have two groups of wavefronts, each with
// every other 32 of the reduction, and half a compute unit's LDS.
//
// What bounds it: the large tiles the matrix cores and the card's power (511 rows of 2,048 x 11,264 1.2 PFLOP/s of bfloat16 products, six for
// each), the small ones what a compute unit takes from L2 (47 GB/s each with 256 tiles).  us of a product, with its split, against the library's
// float32 instructions: 511 rows of 2,048 x 6,144 78 / 96 to 119, x 11,264 123 / 214, 5,632 x 2,048 84 / 92, 300 x 2,048 x 11,264 102 / 144,
// 1,024 x 3,584 x 40,960 1,448 / 2,004.  Error against 64 bits, relative, of 2,048 products of normal numbers 2.8e-7 / 8.1e-7, of
// 5,632 4.7e-7 / 1.3e-6.
#include <algorithm>
#include <type_traits>

#include "lds_loads.h"
#include "split_f32.h"

#define LS_K 32       // numbers of the reduction a stage
#define LS_ROW 192    // bytes of an activation row's stage: 64 of each part
#define LS_UNITS 256  // compute units
// piece p (of eight) of weight row r lies at p ^ ((r >> 1) & 7); piece p (of twelve, four a part) of activation row r at p ^ ((r >> 2) & 3)
__device__ __forceinline__ int ls_weight_at(int row, int piece) { return row * LS_K + ((piece ^ ((row >> 1) & 7)) << 2); }
__device__ __forceinline__ int ls_row_at(int row, int piece) { return row * LS_ROW + ((piece ^ ((row >> 2) & 3)) << 4); }

// WI x XI wavefronts along weight rows and activation rows, each WB x XB blocks of 32 x 32; KG such groups of wavefronts, which multiply a
// KG-th of a stage each (of KG times 32 numbers of the reduction).
template <int WI_, int XI_, int WB_, int XB_, int RING_, int KG_ = 1> struct SplitTile {
  static constexpr int WI = WI_, XI = XI_, WB = WB_, XB = XB_, RING = RING_, KG = KG_, WAVES = KG * WI * XI;
  static constexpr int W = 32 * WB * WI, X = 32 * XB * XI, K = KG * LS_K;
  static constexpr int BYTES = RING * KG * (W * 4 * LS_K + X * LS_ROW);
  static_assert(KG == 1 || W * X * 4 <= BYTES, "the groups' results fit the ring");
  static_assert(BYTES <= 163840, "the ring fits LDS");
  static_assert(KG * X * LS_ROW % (1024 * WAVES) == 0 && KG * W * 4 * LS_K % (1024 * WAVES) == 0, "whole loads for every wavefront");
};

template <typename T, bool NT>
__global__ void __launch_bounds__(64 * T::WAVES)
linear_split_kernel(const float* x, const __bf16* parts, const float* w, float* out, int rows, int n_out, int width, int row_tiles) {
  constexpr int WB = T::WB, XB = T::XB, RING = T::RING, WAVES = T::WAVES;
  constexpr int KG = T::KG;
  constexpr unsigned W1 = T::W * 4 * LS_K, X1 = T::X * LS_ROW, WT = KG * W1, XT = KG * X1;  // bytes of a group's part of a stage, of a stage
  constexpr int NPW = WT / 1024 / WAVES, NPX = XT / 1024 / WAVES, PER = NPW + NPX;  // loads of a wavefront a stage
  __shared__ __attribute__((aligned(1024))) char lds[T::BYTES];
  // the row tiles of a block of weight rows go to one die one after the other, as they read the same weights (see linear_tiled.hip)
  const unsigned die = blockIdx.x & 7, each = gridDim.x >> 3, extra = gridDim.x & 7;
  const unsigned pair = die * each + min(die, extra) + (blockIdx.x >> 3);
  const int block = static_cast<int>(pair / row_tiles), n0 = block * T::W, row0 = static_cast<int>(pair % row_tiles) * T::X;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 31, g = lane >> 5, wi = wave % T::WI, xi = wave / T::WI % T::XI, kg = wave / (T::WI * T::XI);

  // where this lane's pieces of a stage start, in bytes (rows past the end repeat the last one)
  const float* const w_block = w + static_cast<int64_t>(n0) * width;
  unsigned wsrc[NPW], xsrc[NPX];
#pragma unroll
  for (int i = 0; i < NPW; ++i) {
    const int at = 8 * (wave + WAVES * i) + (lane >> 3), r = at % T::W, p = (lane & 7) ^ ((r >> 1) & 7);
    wsrc[i] = 4u * (static_cast<unsigned>(min(r, n_out - 1 - n0)) * static_cast<unsigned>(width) + at / T::W * LS_K) + 16 * p;
  }
#pragma unroll
  for (int i = 0; i < NPX; ++i) {
    const int at = 64 * (wave + WAVES * i) + lane, r = at / 12 % T::X, p = (at % 12) ^ ((r >> 2) & 3);
    xsrc[i] = 6u * static_cast<unsigned>(min(row0 + r, rows - 1)) * static_cast<unsigned>(width) + at / 12 / T::X * LS_ROW + 16 * p;
  }
  // (blocks start the reduction at different stages and wrap round, see moe_tiled_f32.hip)
  const int stages = width / T::K;
  const int rot = width % 256 == 0 ? static_cast<int>(static_cast<unsigned>(block) % static_cast<unsigned>(stages)) : 0;
  auto place = [&](int s) {  // (past the end: the last stage again)
    const int k = min(s, stages - 1) + rot;
    return static_cast<unsigned>(k < stages ? k : k - stages);
  };
  auto load = [&](int buf, int i, unsigned stage) {  // the i-th of a stage's loads
    if (i < NPX) lds_load16<false>(lds, RING * WT + buf * XT + 1024 * (wave + WAVES * i), xsrc[i] + KG * LS_ROW * stage, parts);
    else if (i < PER) lds_load16<NT>(lds, buf * WT + 1024 * (wave + WAVES * (i - NPX)), wsrc[i - NPX] + 4 * T::K * stage, w_block);
  };

  f32x16 large[WB][XB], small[WB][XB];
#pragma unroll
  for (int j = 0; j < WB; ++j)
#pragma unroll
    for (int t = 0; t < XB; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) large[j][t][i] = small[j][t][i] = 0.f;
  int w_at[2][2], x_at[2][3];  // half of the stage; piece of the lane's two, part
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
    for (int p = 0; p < 2; ++p) w_at[kk][p] = 4 * ls_weight_at(m, 4 * kk + 2 * g + p);
#pragma unroll
    for (int p = 0; p < 3; ++p) x_at[kk][p] = ls_row_at(m, 4 * p + 2 * kk + g);
  }
  const char* const ws = lds + kg * W1 + 32 * WB * wi * 4 * LS_K;
  const char* const xs = lds + RING * WT + kg * X1 + 32 * XB * xi * LS_ROW;
  struct Weights { bf16x8 w[WB][3]; };
  struct Half { bf16x8 x[XB][3]; };
  struct Raw { f32x4 a[WB], b[WB]; };
  Half x0, x1;
  Weights w0, w1;
  Raw raw;
  auto read_w = [&](int buf, int kk) {
#pragma unroll
    for (int j = 0; j < WB; ++j) {
      raw.a[j] = *reinterpret_cast<const f32x4*>(ws + buf * WT + 32 * j * 4 * LS_K + w_at[kk][0]);
      raw.b[j] = *reinterpret_cast<const f32x4*>(ws + buf * WT + 32 * j * 4 * LS_K + w_at[kk][1]);
    }
  };
  auto split = [&](Weights& w) {
#pragma unroll
    for (int j = 0; j < WB; ++j) split8(raw.a[j], raw.b[j], w.w[j]);
  };
  auto read_x = [&](Half& h, int buf, int kk) {
#pragma unroll
    for (int t = 0; t < XB; ++t)
#pragma unroll
      for (int p = 0; p < 3; ++p) h.x[t][p] = *reinterpret_cast<const bf16x8*>(xs + buf * XT + 32 * t * LS_ROW + x_at[kk][p]);
  };
  auto products = [&](const Weights& w, const Half& h) {
    auto add = [&](f32x16 (&sum)[WB][XB], int p, int q) {
#pragma unroll
      for (int j = 0; j < WB; ++j)
#pragma unroll
        for (int t = 0; t < XB; ++t) sum[j][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w.w[j][p], h.x[t][q], sum[j][t], 0, 0, 0);
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
    for (int i = 0; i < 6 * WB * XB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x2, (48 * WB + 6 * WB * XB - 1) / (6 * WB * XB), 0);
    }
  };

#pragma unroll
  for (int s = 0; s < RING; ++s)
#pragma unroll
    for (int i = 0; i < PER; ++i) load(s, i, place(s));
  wait_loads<PER * (RING - 1)>();
  lds_barrier();
  int buf = 0;
  read_w(buf, 0);
  read_x(x0, buf, 0);
  split(w0);
  read_w(buf, 1);
  read_x(x1, buf, 1);
  // Stage s, the first half's operands ready, the second half's on their way from LDS; LEFT: at least so many stages follow.
  auto stage = [&](auto left, int s) {
    constexpr int LEFT = decltype(left)::value;
    __builtin_amdgcn_sched_barrier(0);
    products(w0, x0);
    split(w1);
    interleave();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (LEFT > 0) {
      wait_loads<PER * (RING - 2 < LEFT - 1 ? RING - 2 : LEFT - 1)>();  // stage s + 1 has landed
      lds_barrier();
      const int free = buf;  // nobody reads stage s any more
      buf = buf + 1 == RING ? 0 : buf + 1;
      read_w(buf, 0);
      read_x(x0, buf, 0);
      if constexpr (LEFT >= RING) {
        const unsigned next = place(s + RING);
#pragma unroll
        for (int i = 0; i < PER; ++i) load(free, i, next);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    products(w1, x1);
    if constexpr (LEFT > 0) {
      split(w0);
      interleave();
      __builtin_amdgcn_sched_barrier(0);
      read_w(buf, 1);
      read_x(x1, buf, 1);
    }
  };
#define LS_STAGE(LEFT, S) stage(std::integral_constant<int, (LEFT)>{}, (S))
  int s = 0;
  for (; s < stages - RING; ++s) LS_STAGE(RING, s);
  // the last ones, for which everything has been asked for: once the first has let the others go on arriving, all have
  if (s < stages - 1 && stages - 1 - s >= RING - 1) {
    LS_STAGE(RING - 1, s);
    ++s;
  }
  for (; s < stages - 1; ++s) LS_STAGE(1, s);
  LS_STAGE(0, stages - 1);
#undef LS_STAGE
  wait_loads<0>();  // (with fewer stages than the ring holds, the last one again)

#pragma unroll
  for (int j = 0; j < WB; ++j)
#pragma unroll
    for (int t = 0; t < XB; ++t) large[j][t] += small[j][t];
  if constexpr (KG > 1) {  // the groups' sums, in their order
    static_assert(KG == 2, "one other group");
    float* const sums = reinterpret_cast<float*>(lds) + (wave % (T::WI * T::XI)) * (WB * XB * 16 * 64) + lane;
    __syncthreads();
    if (kg > 0)
#pragma unroll
      for (int j = 0; j < WB; ++j)
#pragma unroll
        for (int t = 0; t < XB; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) sums[(16 * (j * XB + t) + i) * 64] = large[j][t][i];
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int j = 0; j < WB; ++j)
#pragma unroll
      for (int t = 0; t < XB; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) large[j][t][i] += sums[(16 * (j * XB + t) + i) * 64];
  }
  // lane holds weight rows n0 + 32 (WB wi + j) + 8 q + 4 g + i of activation row row0 + 32 (XB xi + t) + m
  const bool vec = (n_out & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
  for (int t = 0; t < XB; ++t) {
    const int r = row0 + 32 * (XB * xi + t) + m;
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < WB; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int nb = n0 + 32 * (WB * wi + j) + 8 * q + 4 * g;
        f32x4 v;
        bool numbers = true;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] = large[j][t][4 * q + i];
          numbers = numbers && is_number(v[i]);
        }
        if (!numbers)
#pragma unroll 1
          for (int i = 0; i < 4; ++i)
            if (nb + i < n_out) {
              const float again = plain_dot(x + static_cast<int64_t>(r) * width, w + static_cast<int64_t>(nb + i) * width, width);
              v = i == 0 ? f32x4{again, v[1], v[2], v[3]} : i == 1 ? f32x4{v[0], again, v[2], v[3]}
                : i == 2 ? f32x4{v[0], v[1], again, v[3]} : f32x4{v[0], v[1], v[2], again};
            }
        float* const o = out + static_cast<int64_t>(r) * n_out + nb;
        if (vec && nb + 4 <= n_out) {
          *reinterpret_cast<f32x4*>(o) = v;
          continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nb + i < n_out) o[i] = v[i];
      }
  }
}

// parts [rows, width / 32, 3, 32] of x [rows, width]: a thread eight numbers.
__global__ void __launch_bounds__(256) split_rows_kernel(const float* __restrict__ x, __bf16* __restrict__ parts, int64_t eights) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= eights) return;
  const f32x4 a = *reinterpret_cast<const f32x4*>(x + 8 * i), b = *reinterpret_cast<const f32x4*>(x + 8 * i + 4);
  bf16x8 p[3];
  split8(a, b, p);
  __bf16* const to = parts + i / 4 * 96 + i % 4 * 8;
#pragma unroll
  for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(to + 32 * q) = p[q];
}

namespace {

template <typename T>
int64_t tiles_of(int64_t rows, int64_t n_out) { return ((rows + T::X - 1) / T::X) * ((n_out + T::W - 1) / T::W); }

template <typename T>
int linear_split(const float* x, const void* parts, const float* w, float* out, int64_t rows, int64_t n_out, int64_t width,
                 hipStream_t stream) {
  const int64_t row_tiles = (rows + T::X - 1) / T::X, tiles = tiles_of<T>(rows, n_out);
  IX_REQUIRE(tiles < (int64_t(1) << 31), "too many workgroups for one launch");
#define LAUNCH(NT)                                                                                                       \
  hipLaunchKernelGGL((linear_split_kernel<T, NT>), dim3(static_cast<unsigned>(tiles)), dim3(64 * T::WAVES), 0, stream, x,    \
                     (const __bf16*)parts, w, out, (int)rows, (int)n_out, (int)width, (int)row_tiles)
  if (row_tiles == 1 && (reinterpret_cast<uintptr_t>(w) & 127) == 0) LAUNCH(true);  // (whole lines, read once)
  else LAUNCH(false);
#undef LAUNCH
  return ix_check_launch("ix_linear_split");
}

// by the rows of both kinds that a tile has
using Tile0 = SplitTile<2, 2, 1, 1, 2, 2>;  // 64 x 64, two groups, two workgroups a compute unit
using Tile1 = SplitTile<4, 2, 1, 2, 4>;     // 128 x 128
using Tile2 = SplitTile<6, 2, 1, 2, 3>;     // 192 x 128

// About how long a product takes in tiles T, in us: so much a round of the compute units, and so much for what all of them load and multiply.
template <typename T>
double time_of(int64_t rows, int64_t n_out, int64_t width, double round, double work) {
  const int64_t tiles = tiles_of<T>(rows, n_out);
  return (round * ((tiles + LS_UNITS - 1) / LS_UNITS) + work * tiles / LS_UNITS) * width / 2048;
}

}  // namespace

// x on a 16-byte boundary, in rows of a multiple of 32 numbers; parts: six bytes a number.
extern "C" int ix_split_rows(const float* x, void* parts, int64_t rows, int64_t width, hipStream_t stream) {
  IX_REQUIRE(rows >= 0 && width > 0 && width % LS_K == 0, "rows of a multiple of 32 numbers");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(parts)) & 15) == 0, "operands must lie on 16-byte boundaries");
  const int64_t eights = rows * width / 8, groups = (eights + 255) / 256;
  IX_REQUIRE(groups < (int64_t(1) << 31), "too many workgroups for one launch");
  if (eights == 0) return 0;
  hipLaunchKernelGGL(split_rows_kernel, dim3(static_cast<unsigned>(groups)), dim3(256), 0, stream, x, (__bf16*)parts, eights);
  return ix_check_launch("ix_split_rows");
}

// (a lane's place in its block of weights, and in the activations, is counted in 32 bits of bytes)
static bool small_enough(int64_t rows, int64_t n_out, int64_t width) {
  return 6 * rows * width < (int64_t(1) << 32) && 192 * 4 * width < (int64_t(1) << 32) && n_out < (int64_t(1) << 31) - 512;
}

// The tile for a product, 0 to 2, or -1 where the vendor's library is likely to be as fast: it is taken to form 115 TFLOP/s (110 to 140 with
// many tiles, 20 to 100 with few), the split of the activations to take 5 us.  Over 112 products of 48 to 1,024 rows (2,048 x 6,144, 2,048 x
// 2,048, 2,048 x 11,264, 5,632 x 2,048, 3,584 x 4,608, 3,584 x 3,584, 3,584 x 40,960) the 54 that the line leaves to the tiles take, with the
// split, 0.775 of the library's time (geometric mean; at most 1.02), the others would take 1.27.
extern "C" int ix_linear_split_tile(int64_t rows, int64_t n_out, int64_t width) {
  if (rows <= 0 || n_out <= 0 || width <= 0 || width % (2 * LS_K) != 0 || !small_enough(rows, n_out, width)) return -1;
  const double times[3] = {time_of<Tile0>(rows, n_out, width, 20.0, 7.5), time_of<Tile1>(rows, n_out, width, 55.0, 28.0),
                           time_of<Tile2>(rows, n_out, width, 70.0, 45.0)};
  const int tile = static_cast<int>(std::min_element(times, times + 3) - times);
  return times[tile] + 5.0 < 2.0 * rows * n_out * width / 115e6 ? tile : -1;
}

// Operands on 16-byte boundaries, a width in multiples of 64; parts: `ix_split_rows` of x.  tile: 0 to 2.
extern "C" int ix_linear_split(const float* x, const void* parts, const float* w, float* out, int64_t rows, int64_t n_out, int64_t width,
                               int tile, hipStream_t stream) {
  IX_REQUIRE(rows > 0 && n_out > 0 && width > 0, "sizes must be positive");
  IX_REQUIRE(width % (2 * LS_K) == 0, "the reduction width must be a multiple of 64");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(parts)) & 15) == 0,
             "operands must lie on 16-byte boundaries");
  IX_REQUIRE(small_enough(rows, n_out, width), "sizes too large");
  switch (tile) {
    case 0: return linear_split<Tile0>(x, parts, w, out, rows, n_out, width, stream);
    case 1: return linear_split<Tile1>(x, parts, w, out, rows, n_out, width, stream);
    case 2: return linear_split<Tile2>(x, parts, w, out, rows, n_out, width, stream);
    default: IX_REQUIRE(false, "no such tile"); return 1;
  }
}
