// The gated delta rule over prompt portions, a chunk of 64 rows at a time (delta_rule.hip has the recurrence, its
// operands and the form that walks row by row):
//
//   S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
//
// Within a chunk, with G_i = g_0 .. g_i, the state before it S, and rows of U the u_i / beta_i (so that V enters as it is):
//
//   (I + A) U = V - diag(G) K S,       A_ij = (G_i / G_j) beta_j k_i . k_j  (j < i)
//   O         = diag(G) Q S + P U,     P_ij = (G_i / G_j) beta_j q_i . k_j  (j <= i)
//   S_new     = G_n S + sum_j (G_n / G_j) beta_j k_j u_j^T
//
// so that only U = Uv - W S and S_new are left to the chain over a request's chunks.  Three launches:
//   prepare   a workgroup per (chunk, head): unit rows, the decays, A and P on the matrix cores, the triangular system
//             for Uv and W by blocks of sixteen rows (the four blocks on the diagonal inverted by substitution, the rest
//             matrix products whose results are the next ones' operands as they lie in registers);
//   chain     a workgroup per (request, head, 16 value columns): per chunk two products, W S and K^T U, the state in
//             registers, the next chunk's operands on their way; leaves every chunk its U and the state before it;
//   result    a workgroup per (chunk, head): O.
//
// The generalized delta rule (linear_state.hip has it: a decay w per row and key channel, a correction a (b^T S)),
//
//   S <- diag(w) S - a (b^T S) + k v^T;   o = S^T r
//
// goes the same way with y_i = b_i^T S_(i-1) and, per channel, G_i = w_0 .. w_i: b_i G_(i-1), a_j / G_j, k_j / G_j and
// r_i G_i take the keys' places in
//
//   (I + A) Y = (B G) S + C V,  A_ij = (b_i G_(i-1)) . (a_j / G_j), C_ij with k_j for a_j  (j < i);   U = -Y
//   O = (R G) S + P U + Q V,    P_ij = (r_i G_i) . (a_j / G_j), Q_ij with k_j              (j <= i)
//   S_new = diag(G_n) S + sum_j (G_n / G_j) (a_j u_j^T + k_j v_j^T)
//
// where Q V and the k_j v_j^T, which need no state, are formed by the first launch.  The caller answers for 1 / G_63 being
// a float32 number (a decay no smaller than e^-1).
//
// Everything is held in float32.  The matrix cores' 32-bit sums (v_mfma_f32_16x16x4_f32, in order) are kept to sixteen or 32
// terms each, what is added to a number is summed up before it; the keys' inner products and the state's sums are 64-bit
// (v_mfma_f64_16x16x4_f64), as are the sums of the decays' logarithms, so that the ratio of two late rows is as exact as that
// of two early ones (per channel: the decays' products), and what rows are multiplied by is rounded once.  So results and
// states are no further from the float64 recurrence than row by row: of their norms, 16 requests of 8 heads of 128 x 128, 1.0e-7
// and 0.6e-7 against 1.2e-7 and 0.7e-7 with the quickest decays, 1.5e-7 and 1.0e-7 against 5.8e-7 and 7.3e-7 with slow ones
// (32-bit sums one after the other throughout: 2.4e-7 and 1.5e-7).  The generalized rule, decays e^(-0.61 sigmoid(normal)):
// 0.59e-7 and 0.37e-7 against 0.87e-7 and 0.46e-7 (1.4e-7 and 1.5e-7), slow ones 1.1e-7 and 0.7e-7 against 2.2e-7 and 2.3e-7;
// only where every channel of every row forgets as fast as it can (e^-0.61) the state is 0.36e-7 off against 0.34e-7.
//
// What bounds it: row by row, the chain of dependent sums of a row (0.33 us a row whatever the chip is doing).  In chunks
// the chain is 64 times shorter and its step two small products (3.6 us a chunk).  Measured with 16 heads of 128 x 128, one
// request, all three launches against row by row: 44 against 46 us at 128 rows, 51 against 72 at 200, 68 against 172 at
// 500, 141 against 474 at 1,437, 176 against 672 at 2,048.  The generalized rule, 32 heads
// of 64 x 64: 42 against 43 us at 160 rows, 46 against 66 at 256, 169 against 492 at 2,048 (with 32-bit sums 130).
//
// A lane's operand of a 16 x 16 x 4 product is one number of row (column) l % 16 at reduction index l / 16.  Operands
// are read four numbers at a time, index 16 s + 4 (l / 16) + e, and the e-th of them meet in one instruction.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4), aligned(16)));

#define DC_ROWS 64
#define DC_THREADS 256

// where the parts of a (chunk, head) lie in its block of the workspace, in floats
struct DeltaBlock {
  int dim, vdim, more;  // more: the generalized rule
  __host__ __device__ __forceinline__ int64_t w() const { return 0; }                          // [64][dim]: -W
  __host__ __device__ __forceinline__ int64_t kt() const { return 64 * dim; }                  // [dim][64]: k_j, or (G_n / G_j) a_j
  __host__ __device__ __forceinline__ int64_t q() const { return 128 * dim; }                  // [64][dim]: G_i q_i
  __host__ __device__ __forceinline__ int64_t p() const { return 192 * dim; }                  // [64][64]: P, tiles j <= i
  __host__ __device__ __forceinline__ int64_t u() const { return 192 * dim + 4096; }           // [vdim][64]: Uv, then U
  __host__ __device__ __forceinline__ int64_t s() const { return u() + 64 * vdim; }            // [vdim][dim]: S before
  __host__ __device__ __forceinline__ int64_t g() const { return s() + static_cast<int64_t>(dim) * vdim; }  // [dim]: G_n
  __host__ __device__ __forceinline__ int64_t m() const { return g() + dim; }  // [vdim][dim] double: sum_j (G_n / G_j) k_j v_j^T
  __host__ __device__ __forceinline__ int64_t rest() const { return m(); }  // [64] double: (G_n / G_j) beta_j (the gated rule)
  __host__ __device__ __forceinline__ int64_t size() const { return m() + (more ? 2 * static_cast<int64_t>(dim) * vdim : 128); }
};

__device__ __forceinline__ f32x4 dc_mac(f32x4 a, f32x4 b, f32x4 acc) {
#pragma unroll
  for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
  return acc;
}

// The same with 64-bit sums (v_mfma_f64_16x16x4_f64, half the rate).  Its result e of a lane is row 4 e + l / 16: with the
// first operand's rows handed over in the order of `dc_turn` a lane has the rows 4 (l / 16) + e, as in 32 bits.
__device__ __forceinline__ int dc_turn(int m) { return 4 * (m & 3) + (m >> 2); }
__device__ __forceinline__ f64x4 dc_mac64(f32x4 a, f32x4 b, f64x4 acc) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a[e]), static_cast<double>(b[e]), acc, 0, 0, 0);
  return acc;
}
// e^c, c <= 0, without the rounding of c
__device__ __forceinline__ float dc_exp(double c) {
  const float hi = static_cast<float>(c), e = expf(hi);
  return fmaf(e, static_cast<float>(c - hi), e);
}

// Numbers that are not finite stay with their row and the later ones, as row by row.  A triangular block of sixteen rows
// keeps zeros for the rows that a row does not see, but zero times NaN is NaN: where a block's operand holds such numbers,
// it is multiplied without them, and the results that see one of them become NaN.  `seen`: this lane's numbers of a matrix
// that holds 1 where the triangle does.
__device__ __forceinline__ bool dc_odd(const f32x4 x) {  // is any of them not finite?  (the products are 0 or NaN)
  return !(x[0] * 0.f + x[1] * 0.f + (x[2] * 0.f + x[3] * 0.f) == 0.f);
}
__device__ __forceinline__ f32x4 dc_seen(int row, int first, bool own) {  // rows first + e that `row` sees, its own with `own`
  f32x4 s;
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = first + e < row + (own ? 1 : 0) ? 1.f : 0.f;
  return s;
}
// the operand x without its numbers that are not finite, and where they were
__device__ __forceinline__ void dc_part(const f32x4 x, f32x4& clean, f32x4& odd) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bool bad = !(x[e] * 0.f == 0.f);
    clean[e] = bad ? 0.f : x[e];
    odd[e] = bad ? 1.f : 0.f;
  }
}
__device__ __forceinline__ f32x4 dc_spoil(const f32x4 x, const f32x4 count) {
  f32x4 y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = count[e] > 0.f ? __builtin_nanf("") : x[e];
  return y;
}
// acc + the product of a triangular block with x: the block is the first operand, or the second one
__device__ __forceinline__ f32x4 dc_mac_block(f32x4 block, f32x4 x, f32x4 seen, f32x4 acc) {
  const f32x4 none = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 clean, odd;
  dc_part(x, clean, odd);
  return dc_spoil(dc_mac(block, clean, acc), dc_mac(seen, odd, none));
}
__device__ __forceinline__ f64x4 dc_mac64_block(f32x4 block, f32x4 x, f32x4 seen, f64x4 acc) {  // (the block's rows in the order of `dc_turn`)
  const f32x4 none = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 clean, odd;
  dc_part(x, clean, odd);
  acc = dc_mac64(block, clean, acc);
  const f32x4 count = dc_mac(seen, odd, none);
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = count[e] > 0.f ? __builtin_nan("") : acc[e];
  return acc;
}
__device__ __forceinline__ f32x4 dc_narrow(const f64x4 x) {
  return f32x4{static_cast<float>(x[0]), static_cast<float>(x[1]), static_cast<float>(x[2]), static_cast<float>(x[3])};
}
__device__ __forceinline__ f32x4 dc_mac_block_second(f32x4 x, f32x4 block, f32x4 seen, f32x4 acc) {
  const f32x4 none = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 clean, odd;
  dc_part(x, clean, odd);
  return dc_spoil(dc_mac(clean, block, acc), dc_mac(odd, seen, none));
}

// A (in LDS, strictly lower) -> the inverses of the blocks on the diagonal of I + A, less I; one wavefront, lane (block, column)
template <int LA>
__device__ __forceinline__ void dc_invert_diagonal(const float* a_s, float (*t_s)[16][20], int b, int col) {
  float x[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float s = i == col ? 1.f : 0.f;
    const float* ar = a_s + (16 * b + i) * LA + 16 * b;
#pragma unroll
    for (int j = 0; j < i; ++j) s = fmaf(-ar[j], x[j], s);
    x[i] = s;
    if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (not all of the block's numbers at once: that would be 120 registers)
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) t_s[b][i][col] = i == col ? 0.f : x[i];
}

// x <- (I + A)^-1 x for NT tiles of sixteen columns: [tile][block of sixteen rows], a lane's numbers rows 4 g + e of column m.
// What is added to a row is summed up by itself, sixteen terms at a time, and rounds at its own size.
template <int LA, int NT>
__device__ __forceinline__ void dc_solve(const float* a_s, const float (*t_s)[16][20], int m, int g, f32x4 (&x)[NT][4]) {
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    f32x4 sum[NT];
#pragma unroll
    for (int a = 0; a < b; ++a) {
      const f32x4 na = -*reinterpret_cast<const f32x4*>(a_s + (16 * b + m) * LA + 16 * a + 4 * g);
      f32x4 part[NT];
#pragma unroll
      for (int u = 0; u < NT; ++u) part[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int u = 0; u < NT; ++u) part[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(na[e], x[u][a][e], part[u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < NT; ++u) sum[u] = a == 0 ? part[u] : sum[u] + part[u];
    }
    if (b > 0) {
#pragma unroll
      for (int u = 0; u < NT; ++u) x[u][b] += sum[u];
    }
    const f32x4 inv = *reinterpret_cast<const f32x4*>(&t_s[b][m][4 * g]);
    f32x4 y[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) y[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    bool odd = false;
#pragma unroll
    for (int u = 0; u < NT; ++u) odd = odd || dc_odd(x[u][b]);
    if (__any(odd)) {
#pragma unroll
      for (int u = 0; u < NT; ++u) y[u] = dc_mac_block(inv, x[u][b], dc_seen(m, 4 * g, false), y[u]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int u = 0; u < NT; ++u) y[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(inv[e], x[u][b][e], y[u], 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < NT; ++u) x[u][b] += y[u];
    __builtin_amdgcn_sched_barrier(0);  // (the next block's operands: not before)
  }
}

// A chunk and head takes a workgroup some 30 us whatever else the chip is doing (sums and inner products one behind the other), so
// three of them share a compute unit: rows stay in LDS as they came, with their factors beside them, and a wavefront solves for
// two tiles at a time.  All three launches, us, with two workgroups to a compute unit (rows in 32 bits, four tiles) / as it is: 16
// heads of 128 x 128, 33 chunks of two requests (528 workgroups, 16 more than went at once) 178 / 160, 32 of one 184 / 176, 16
// requests of 300 rows 356 / 298.  A lane has 168 registers so and needs 132.
template <int DIM>
__global__ void __launch_bounds__(DC_THREADS, 3)
delta_chunks_prepare_kernel(const bf16_t* q, const bf16_t* k, const bf16_t* v, int64_t q_stride, int64_t k_stride,
                            int64_t v_stride, const float* __restrict__ ab, const float* __restrict__ a_log,
                            const float* __restrict__ dt_bias, const int32_t* __restrict__ chunk_row0,
                            const int32_t* __restrict__ chunk_rows, float* __restrict__ work, int heads, int kv_heads,
                            int vdim) {
  constexpr int LD = DIM + 8, LA = DC_ROWS + 4;
  // Rows as they came, and the factors that make them unit rows: half the room of the products.
  __shared__ __attribute__((aligned(16))) bf16_t k_s[DC_ROWS * LD];
  // the queries, and once they are done with A in their place
  __shared__ __attribute__((aligned(16))) unsigned char qa_s[DC_ROWS * (2 * LD > 4 * LA ? 2 * LD : 4 * LA)];
  bf16_t* const q_s = reinterpret_cast<bf16_t*>(qa_s);
  float* const a_s = reinterpret_cast<float*>(qa_s);
  __shared__ float f_s[2][DC_ROWS];  // the keys' factors, the queries'
  __shared__ __attribute__((aligned(16))) float t_s[4][16][20];  // inverses of the blocks on the diagonal of I + A
  __shared__ double c_s[DC_ROWS];                                // log G_i
  __shared__ double beta_s[DC_ROWS], g_s[DC_ROWS], rest_s[DC_ROWS];  // beta_i, G_i, G_n / G_i (products with them round once)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int head = blockIdx.x, chunk = blockIdx.y;
  const int kv = head / (heads / kv_heads);
  const int64_t row0 = chunk_row0[chunk];
  const int n = chunk_rows[chunk];
  const DeltaBlock blk{DIM, vdim, 0};
  float* mine = work + (static_cast<int64_t>(chunk) * heads + head) * blk.size();

  // ---- unit rows into LDS: four threads a row, a quarter of its numbers each; rows past the chunk's end are zeros
  {
    constexpr int QUARTER = DIM / 4;
    const int row = tid >> 2, part = tid & 3;
    const int64_t src = row0 + min(row, n - 1);
    const bf16_t* rows[2] = {k + src * k_stride + kv * DIM + part * QUARTER, q + src * q_stride + kv * DIM + part * QUARTER};
    uint4 raw[2][QUARTER / 8];
#pragma unroll
    for (int which = 0; which < 2; ++which)
#pragma unroll
      for (int i = 0; i < QUARTER / 8; ++i) raw[which][i] = *reinterpret_cast<const uint4*>(rows[which] + 8 * i);
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      bf16_t* dst = (which ? q_s : k_s) + row * LD + part * QUARTER;
      double sum = 0.;  // (a row's factor is one error for all its numbers)
#pragma unroll
      for (int i = 0; i < QUARTER / 8; ++i) {
        const uint32_t u[4] = {raw[which][i].x, raw[which][i].y, raw[which][i].z, raw[which][i].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const double lo = __uint_as_float(u[e] << 16), hi = __uint_as_float(u[e] & 0xffff0000u);
          sum += lo * lo;
          sum += hi * hi;
        }
        *reinterpret_cast<uint4*>(dst + 8 * i) = raw[which][i];
      }
      float ss = static_cast<float>(sum);
      ss += ix_dpp<IX_DPP_XOR1>(ss);
      ss += ix_dpp<IX_DPP_XOR2>(ss);
      if (part == 0)
        f_s[which][row] = row < n ? (which ? 1.0f / sqrtf(static_cast<float>(DIM)) : 1.0f) / sqrtf(ss + 1e-6f) : 0.f;
    }
  }
  if (wave == 0) {
    const bool live = lane < n;
    const int64_t row = row0 + min(lane, n - 1);
    const float x = ab[row * 2 * heads + head] + dt_bias[head];
    float lg = live ? -expf(a_log[head]) * (x > 20.f ? x : log1pf(expf(x))) : 0.f;
    // (a decay of e^-200 is zero in float32; below that, and at minus infinity, the differences of the sums, which are the
    // ratios of the rows that come after, would lose those rows' own logarithms.  NaN stays.)
    if (lg < -200.f) lg = -200.f;
    double c = lg;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double below = __shfl_up(c, off, 64);
      if (lane >= off) c += below;
    }
    const double last = __shfl(c, 63, 64);
    c_s[lane] = c;
    g_s[lane] = exp(c);
    rest_s[lane] = exp(last - c);
    beta_s[lane] = live ? 1.0f / (1.0f + expf(-ab[row * 2 * heads + heads + head])) : 0.f;
  }
  __syncthreads();

  // four numbers of a unit row
  auto unit4 = [&](const bf16_t* at, float f) {
    const uint2 u = *reinterpret_cast<const uint2*>(at);
    return f32x4{__uint_as_float(u.x << 16) * f, __uint_as_float(u.x & 0xffff0000u) * f, __uint_as_float(u.y << 16) * f,
                 __uint_as_float(u.y & 0xffff0000u) * f};
  };
  // ---- q_i . k_j, then k_i . k_j: the ten tiles on and below the diagonal of each
  auto score = [&](const bf16_t* rows, const float* factors, int pair, auto&& put) {
    const int rt = pair < 1 ? 0 : (pair < 3 ? 1 : (pair < 6 ? 2 : 3)), ct = pair - rt * (rt + 1) / 2;
    const bf16_t* ar = rows + (16 * rt + dc_turn(m)) * LD + 4 * g;
    const bf16_t* br = k_s + (16 * ct + m) * LD + 4 * g;
    const float fa = factors[16 * rt + dc_turn(m)], fb = f_s[0][16 * ct + m];
    f64x4 s0 = f64x4{0., 0., 0., 0.}, s1 = s0;
#pragma unroll
    for (int c = 0; c < DIM / 16; c += 2) {
      s0 = dc_mac64(unit4(ar + 16 * c, fa), unit4(br + 16 * c, fb), s0);
      s1 = dc_mac64(unit4(ar + 16 * c + 16, fa), unit4(br + 16 * c + 16, fb), s1);
    }
    const int j = 16 * ct + m;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 16 * rt + 4 * g + e;
      const float ratio = dc_exp(fmin(c_s[i] - c_s[j], 0.0));  // (above the diagonal: not used)
      put(i, j, ratio * (s0[e] + s1[e]));
    }
  };
#pragma unroll 1
  for (int pair = wave; pair < 10; pair += 4)
    score(q_s, f_s[1], pair, [&](int i, int j, double x) { mine[blk.p() + i * 64 + j] = j <= i ? static_cast<float>(beta_s[j] * x) : 0.f; });
  // ---- what the chain and the result take as they are
  for (int id = tid; id < DIM * 16; id += DC_THREADS) {
    const int row = id / (DIM / 4), d = 4 * (id % (DIM / 4));
    f32x4 x = unit4(q_s + row * LD + d, f_s[1][row]);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = static_cast<float>(x[e] * g_s[row]);
    *reinterpret_cast<f32x4*>(mine + blk.q() + row * DIM + d) = x;
  }
  __syncthreads();
#pragma unroll 1
  for (int pair = 3 - wave; pair < 10; pair += 4)  // (the wavefronts that had three tiles above have two)
    score(k_s, f_s[0], pair, [&](int i, int j, double x) { a_s[i * LA + j] = j < i ? static_cast<float>(beta_s[j] * x) : 0.f; });
  for (int id = tid; id < DIM * 16; id += DC_THREADS) {
    const int d = id >> 4, jq = 4 * (id & 15);
    f32x4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = ix_load(k_s + (jq + e) * LD + d) * f_s[0][jq + e];
    *reinterpret_cast<f32x4*>(mine + blk.kt() + d * 64 + jq) = x;
  }
  if (tid < DC_ROWS) reinterpret_cast<double*>(mine + blk.rest())[tid] = rest_s[tid] * beta_s[tid];
  for (int d = tid; d < DIM; d += DC_THREADS) mine[blk.g() + d] = static_cast<float>(g_s[DC_ROWS - 1]);
  __syncthreads();

  // a wavefront's first tiles of V are asked for before W's, behind which they arrive
  const int tiles = (DIM + vdim) / 16;
  auto ask_v = [&](int t0, unsigned short (&x)[2][4][4]) {
    // (hidden: the rows' places would otherwise be kept in registers from one time to the next, twenty of them in scratch memory)
    int ln = lane;
    asm volatile("" : "+v"(ln));
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bf16_t* from = v + row0 * v_stride + head * vdim + 16 * min(t0 + u, tiles - 1) - DIM + (ln & 15);
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[u][b][e] = from[min(16 * b + 4 * (ln >> 4) + e, n - 1) * v_stride].bits;
    }
  };
  // ---- the diagonal blocks' inverses: lane (block, column), sixteen steps of substitution
  if (wave == 0) dc_invert_diagonal<LA>(a_s, t_s, g, m);
  __builtin_amdgcn_sched_barrier(0);
  unsigned short vx[2][4][4];
  const int v0 = 2 * wave + (DIM / 16 - 2 * wave + 7) / 8 * 8;  // the first of its tiles that are V's
  if (v0 < tiles) ask_v(v0, vx);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();

  // ---- (I + A) [W | Uv] = [diag(G) K | V], two tiles of sixteen columns at a time and wavefront (with four
  // a compute unit's registers hold two workgroups)
#pragma unroll 1
  for (int t0 = 2 * wave; t0 < tiles; t0 += 8) {
    f32x4 x[2][4];  // [tile][block of rows]
    if (16 * t0 < DIM) {  // (DIM / 16 is even: both tiles are W's or both V's)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = 16 * b + 4 * g + e;
            x[u][b][e] = static_cast<float>(g_s[row] * (ix_load(k_s + row * LD + 16 * (t0 + u) + m) * f_s[0][row]));
          }
    } else {
      if (t0 != v0) ask_v(t0, vx);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) x[u][b][e] = ix_bf16_to_f32(vx[u][b][e]);
    }
    dc_solve<LA, 2>(a_s, t_s, m, g, x);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = t0 + u;
      if (t >= tiles) continue;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (16 * t < DIM) {
#pragma unroll
          for (int e = 0; e < 4; ++e) mine[blk.w() + (16 * b + 4 * g + e) * DIM + 16 * t + m] = -x[u][b][e];
        } else {
          *reinterpret_cast<f32x4*>(mine + blk.u() + (16 * t - DIM + m) * 64 + 16 * b + 4 * g) = x[u][b];
        }
      }
    }
  }
}

// The generalized rule's first launch.  w, a, b float32 [T, heads * DIM]; r, k, v bfloat16 rows.
template <int DIM>
__global__ void __launch_bounds__(DC_THREADS, DIM <= 64 ? 2 : 1)
general_chunks_prepare_kernel(const bf16_t* r, const bf16_t* k, const bf16_t* v, int64_t r_stride, int64_t k_stride,
                              int64_t v_stride, const float* __restrict__ w_rows, const float* __restrict__ a_rows,
                              const float* __restrict__ b_rows, const int32_t* __restrict__ chunk_row0,
                              const int32_t* __restrict__ chunk_rows, float* __restrict__ work, float* __restrict__ out,
                              int heads, int vdim) {
  constexpr int LD = (DIM > DC_ROWS ? DIM : DC_ROWS) + 4;  // (a buffer also holds 64 x 64 scores)
  constexpr int SEG = DIM / 4;                             // rows per thread: 256 / DIM threads share a channel
  __shared__ __attribute__((aligned(16))) float x_s[4][DC_ROWS * LD];  // b G, a / G (then A), k / G (then C), r G (then Q)
  __shared__ __attribute__((aligned(16))) float t_s[4][16][20];
  __shared__ double seg_s[DC_THREADS / DIM][DIM];
  __shared__ double gn_s[DIM];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int head = blockIdx.x, chunk = blockIdx.y;
  const int64_t row0 = chunk_row0[chunk];
  const int n = chunk_rows[chunk];
  const DeltaBlock blk{DIM, vdim, 1};
  float* mine = work + (static_cast<int64_t>(chunk) * heads + head) * blk.size();
  float *const b_s = x_s[0], *const a_s = x_s[1], *const k_s = x_s[2], *const r_s = x_s[3];

  // ---- the decays' products down the rows, and the four operands scaled by them (everything is asked for before the first
  // use and under no condition: loads that a condition guards come one after the other, 18 against 26 us for one chunk)
  {
    constexpr int PART = SEG < 16 ? SEG : 16;  // rows whose numbers are asked for together
    const int d = tid % DIM, seg = tid / DIM;
    const int64_t c = static_cast<int64_t>(head) * DIM + d, wide = static_cast<int64_t>(heads) * DIM;
    auto at = [&](int i) { return row0 + min(seg * SEG + i, n - 1); };
    float w[SEG];
#pragma unroll
    for (int i = 0; i < SEG; ++i) w[i] = w_rows[at(i) * wide + c];
    float av[PART], bv[PART], kv[PART], rv[PART];
    auto ask = [&](int i0) {
#pragma unroll
      for (int i = 0; i < PART; ++i) {
        const int64_t t = at(i0 + i);
        av[i] = a_rows[t * wide + c];
        bv[i] = b_rows[t * wide + c];
        kv[i] = ix_load(k + t * k_stride + c);
        rv[i] = ix_load(r + t * r_stride + c);
      }
    };
    ask(0);
    __builtin_amdgcn_sched_barrier(0);
    double p = 1.0;
#pragma unroll
    for (int i = 0; i < SEG; ++i) {
      w[i] = seg * SEG + i < n ? w[i] : 1.0f;
      p *= w[i];
    }
    seg_s[seg][d] = p;
    __syncthreads();
    double all = 1.0;  // G_n
    p = 1.0;
#pragma unroll
    for (int s = 0; s < DC_THREADS / DIM; ++s) {
      p *= s < seg ? seg_s[s][d] : 1.0;
      all *= seg_s[s][d];
    }
    f32x4 kt;
#pragma unroll
    for (int i0 = 0; i0 < SEG; i0 += PART) {
      if (i0 > 0) ask(i0);
#pragma unroll
      for (int i = 0; i < PART; ++i) {
        const int row = seg * SEG + i0 + i;
        const bool live = row < n;  // (one rounding each: the products are 64-bit)
        b_s[row * LD + d] = live ? static_cast<float>(bv[i] * p) : 0.f;
        p *= w[i0 + i];
        const double over = 1.0 / p;
        a_s[row * LD + d] = live ? static_cast<float>(av[i] * over) : 0.f;
        k_s[row * LD + d] = live ? static_cast<float>(kv[i] * over) : 0.f;
        const float rg = live ? static_cast<float>(rv[i] * p) : 0.f;
        r_s[row * LD + d] = rg;
        mine[blk.q() + row * DIM + d] = rg;
        kt[i & 3] = live ? static_cast<float>(av[i] * (all * over)) : 0.f;
        if ((i & 3) == 3) *reinterpret_cast<f32x4*>(mine + blk.kt() + d * 64 + row - 3) = kt;
      }
    }
    if (seg == 0) {
      gn_s[d] = all;
      mine[blk.g() + d] = static_cast<float>(all);
    }
  }
  __syncthreads();

  // ---- the four score matrices, ten tiles on and below the diagonal each: P to the workspace, the others into registers
  // (at most three tiles of each a wavefront) until their operands' buffers are free
  auto score = [&](const float* left, const float* right, int pair, int& rt, int& ct) {
    rt = pair < 1 ? 0 : (pair < 3 ? 1 : (pair < 6 ? 2 : 3));
    ct = pair - rt * (rt + 1) / 2;
    const float* ar = left + (16 * rt + dc_turn(m)) * LD + 4 * g;
    const float* br = right + (16 * ct + m) * LD + 4 * g;
    f64x4 s0 = f64x4{0., 0., 0., 0.}, s1 = s0;
#pragma unroll
    for (int c = 0; c < DIM / 16; c += 2) {
      s0 = dc_mac64(*reinterpret_cast<const f32x4*>(ar + 16 * c), *reinterpret_cast<const f32x4*>(br + 16 * c), s0);
      s1 = dc_mac64(*reinterpret_cast<const f32x4*>(ar + 16 * c + 16), *reinterpret_cast<const f32x4*>(br + 16 * c + 16), s1);
    }
    return dc_narrow(s0 + s1);
  };
  f32x4 qv[3], av[3], cv[3];
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const int pair = wave + 4 * u, back = 3 - wave + 4 * u;  // (who has three tiles of two matrices has two of the others)
    int rt, ct;
    if (pair < 10) {
      const f32x4 s = score(r_s, a_s, pair, rt, ct);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * rt + 4 * g + e, j = 16 * ct + m;
        mine[blk.p() + i * 64 + j] = j <= i ? s[e] : 0.f;
      }
      av[u] = score(b_s, a_s, pair, rt, ct);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (back < 10) {
      qv[u] = score(r_s, k_s, back, rt, ct);
      cv[u] = score(b_s, k_s, back, rt, ct);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // ---- what k and v alone add to the state, a wavefront per tile of value columns
  const int vtiles = vdim / 16;
  auto load_v = [&](int t, f32x4 (&x)[4]) {
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * b + 4 * g + e;
        x[b][e] = ix_load(v + (row0 + min(row, n - 1)) * v_stride + head * vdim + 16 * t + m);  // (past the end: times 0)
      }
  };
#pragma unroll 1
  for (int t = wave; t < vtiles; t += 4) {
    f32x4 x[4];
    load_v(t, x);
#pragma unroll 1
    for (int dt = 0; dt < DIM / 16; ++dt) {
      f64x4 s = f64x4{0., 0., 0., 0.};
      const int d = 16 * dt + dc_turn(m);
      const double gn = gn_s[d];
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          s = __builtin_amdgcn_mfma_f64_16x16x4f64(k_s[(16 * b + 4 * g + e) * LD + d] * gn, static_cast<double>(x[b][e]), s, 0, 0, 0);
      *reinterpret_cast<f64x4*>(reinterpret_cast<double*>(mine + blk.m()) + static_cast<int64_t>(16 * t + m) * DIM + 16 * dt + 4 * g) = s;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const int pair = wave + 4 * u, back = 3 - wave + 4 * u;
    auto place = [&](int pr, float* to, const f32x4& s, bool diagonal) {
      const int rt = pr < 1 ? 0 : (pr < 3 ? 1 : (pr < 6 ? 2 : 3)), ct = pr - rt * (rt + 1) / 2;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * rt + 4 * g + e, j = 16 * ct + m;
        to[i * LD + j] = (j < i || (diagonal && j == i)) ? s[e] : 0.f;
      }
    };
    if (pair < 10) place(pair, a_s, av[u], false);
    if (back < 10) {
      place(back, k_s, cv[u], false);
      place(back, r_s, qv[u], true);
    }
  }
  __syncthreads();
  if (wave == 0) dc_invert_diagonal<LD>(a_s, t_s, g, m);
  __syncthreads();

  // ---- -W = -(I + A)^-1 (B G)
#pragma unroll 1
  for (int t = wave; t < DIM / 16; t += 4) {
    f32x4 x[1][4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[0][b][e] = b_s[(16 * b + 4 * g + e) * LD + 16 * t + m];
    dc_solve<LD, 1>(a_s, t_s, m, g, x);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) mine[blk.w() + (16 * b + 4 * g + e) * DIM + 16 * t + m] = -x[0][b][e];
  }
  // ---- Q V into the result, -(I + A)^-1 C V into U's place
#pragma unroll 1
  for (int t = wave; t < vtiles; t += 4) {
    f32x4 x[4], z[1][4];
    load_v(t, x);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f64x4 o = f64x4{0., 0., 0., 0.}, c = o;
#pragma unroll
      for (int a = 0; a <= b; ++a) {
        const f32x4 ra = *reinterpret_cast<const f32x4*>(r_s + (16 * b + dc_turn(m)) * LD + 16 * a + 4 * g);
        const f32x4 ka = *reinterpret_cast<const f32x4*>(k_s + (16 * b + dc_turn(m)) * LD + 16 * a + 4 * g);
        if (a == b && __any(dc_odd(x[a]))) {
          o = dc_mac64_block(ra, x[a], dc_seen(m, 4 * g, true), o);
          c = dc_mac64_block(ka, x[a], dc_seen(m, 4 * g, false), c);
        } else {
          o = dc_mac64(ra, x[a], o);
          c = dc_mac64(ka, x[a], c);
        }
      }
      z[0][b] = -dc_narrow(c);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * b + 4 * g + e;
        if (row < n) out[((row0 + row) * heads + head) * vdim + 16 * t + m] = static_cast<float>(o[e]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    dc_solve<LD, 1>(a_s, t_s, m, g, z);
#pragma unroll
    for (int b = 0; b < 4; ++b) *reinterpret_cast<f32x4*>(mine + blk.u() + (16 * t + m) * 64 + 16 * b + 4 * g) = z[0][b];
  }
}

// request blockIdx.z's chunks [first, first + count) one after the other, value columns 16 blockIdx.y ..  The state's sums are
// 64-bit: row by row the state is left with fewer roundings than 32-bit sums over a chunk have, 0.8e-7 of its norm after
// quick decays against 0.9e-7 (the generalized rule's, whose terms cancel, 0.5e-7 against 1.8e-7); they cost a chunk's step
// 3.6 instead of 2.8 us.
template <int DIM, bool MORE>
__global__ void __launch_bounds__(DC_THREADS)
delta_chunks_chain_kernel(float* work, const int32_t* __restrict__ seq_ids, const int32_t* __restrict__ seq_first,
                          const int32_t* __restrict__ seq_count, const int32_t* __restrict__ state_slots,
                          float* __restrict__ state, int64_t state_stride, int heads, int vdim) {
  constexpr int LD = DIM + 4, LU = DC_ROWS + 2;
  constexpr int TILES = DIM / 16;                  // tiles of sixteen rows of the state
  constexpr int TS = TILES >= 4 ? TILES / 4 : 1;   // ... per wavefront (with two tiles in all two wavefronts have none)
  __shared__ __attribute__((aligned(16))) float s_s[16 * LD];
  __shared__ __attribute__((aligned(16))) double u_s[16 * LU];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4;
  // (heads first: workgroups go to the chip's eight dies in turn, so a head's column blocks, which read the same W and
  // K^T, share a die's L2 where the heads come in eights: 67 against 70 us at 1,437 rows)
  const int head = blockIdx.x, seq = blockIdx.z;
  const int col = 16 * blockIdx.y + m;
  const int first = seq_first[seq], count = seq_count[seq];
  if (count <= 0) return;
  const bool owns = wave * TS < TILES;
  const DeltaBlock blk{DIM, vdim, MORE};
  const int64_t size = blk.size(), step = heads * size;
  float* at0 = work + (static_cast<int64_t>(first) * heads + head) * size;
  float* sp = state + static_cast<int64_t>(state_slots[seq_ids[seq]]) * state_stride +
              (static_cast<int64_t>(head) * vdim + col) * DIM;
  int row[TS];  // this lane's four rows of the state in each of its tiles
  f32x4 st[TS];
#pragma unroll
  for (int t = 0; t < TS; ++t) {
    row[t] = owns ? 16 * (wave * TS + t) + 4 * g : 0;
    st[t] = *reinterpret_cast<const f32x4*>(sp + row[t]);
  }
  struct Operands { f32x4 w[TILES], kt[TS][4], u, gn[TS]; f64x4 more[MORE ? TS : 1]; };  // more: M, or (G_n / G_j) beta_j
  auto ask = [&](const float* p, Operands& o) {
#pragma unroll
    for (int c = 0; c < TILES; ++c)
      o.w[c] = *reinterpret_cast<const f32x4*>(p + blk.w() + (16 * wave + m) * DIM + 16 * c + 4 * g);
#pragma unroll
    for (int t = 0; t < TS; ++t) {
      const int d = (owns ? 16 * (wave * TS + t) : 0) + dc_turn(m);
#pragma unroll
      for (int s = 0; s < 4; ++s) o.kt[t][s] = *reinterpret_cast<const f32x4*>(p + blk.kt() + d * 64 + 16 * s + 4 * g);
      o.gn[t] = *reinterpret_cast<const f32x4*>(p + blk.g() + row[t]);
      if constexpr (MORE) o.more[t] = *reinterpret_cast<const f64x4*>(reinterpret_cast<const double*>(p + blk.m()) + static_cast<int64_t>(col) * DIM + row[t]);
    }
    o.u = *reinterpret_cast<const f32x4*>(p + blk.u() + col * 64 + 16 * wave + 4 * g);
    if constexpr (!MORE) o.more[0] = *reinterpret_cast<const f64x4*>(reinterpret_cast<const double*>(p + blk.rest()) + 16 * wave + 4 * g);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto work_chunk = [&](float* p, const Operands& o) {
    if (owns) {
#pragma unroll
      for (int t = 0; t < TS; ++t) {
        *reinterpret_cast<f32x4*>(s_s + m * LD + row[t]) = st[t];
        *reinterpret_cast<f32x4*>(p + blk.s() + static_cast<int64_t>(col) * DIM + row[t]) = st[t];
      }
    }
    __syncthreads();
    // (all of a product's operands are asked for before the first is used: left to itself the compiler takes them two by
    // two and waits for each pair)
    f32x4 b[TILES];
#pragma unroll
    for (int c = 0; c < TILES; ++c) b[c] = *reinterpret_cast<const f32x4*>(s_s + m * LD + 16 * c + 4 * g);
    __builtin_amdgcn_sched_barrier(0);
    constexpr int PARTS = TILES < 4 ? TILES : 4;
    f32x4 part[PARTS];
#pragma unroll
    for (int i = 0; i < PARTS; ++i) part[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < TILES; c += PARTS)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < PARTS; ++i)
          part[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[c + i][e], b[c + i][e], part[i], 0, 0, 0);
    f32x4 ws = part[0] + part[1], u;
    if constexpr (PARTS == 4) ws += part[2] + part[3];
    f64x4 us;  // (the state takes U, and what its rows are multiplied by, unrounded)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      us[e] = static_cast<double>(ws[e]) + static_cast<double>(o.u[e]);
      u[e] = static_cast<float>(us[e]);
      if constexpr (!MORE) us[e] *= o.more[0][e];
    }
    *reinterpret_cast<f64x4*>(u_s + m * LU + 16 * wave + 4 * g) = us;
    *reinterpret_cast<f32x4*>(p + blk.u() + col * 64 + 16 * wave + 4 * g) = u;
    f64x4 sum[2];  // two tiles' sums, or the halves of one's
#pragma unroll
    for (int t = 0; t < TS; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sum[t][e] = static_cast<double>(st[t][e]) * static_cast<double>(o.gn[t][e]);
        if constexpr (MORE) sum[t][e] += o.more[t][e];
      }
    if constexpr (TS == 1) sum[1] = f64x4{0., 0., 0., 0.};
    __syncthreads();
    f64x4 bu[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) bu[s] = *reinterpret_cast<const f64x4*>(u_s + m * LU + 16 * s + 4 * g);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < TS; ++t) {
          f64x4& to = sum[TS == 1 ? s & 1 : t];
          to = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(o.kt[t][s][e]), bu[s][e], to, 0, 0, 0);
        }
#pragma unroll
    for (int t = 0; t < TS; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) st[t][e] = static_cast<float>(TS == 1 ? sum[0][e] + sum[1][e] : sum[t][e]);
  };
  Operands one, two;  // the next chunk's operands on their way while this one is worked
  ask(at0, one);
  for (int c = 0; c < count; c += 2) {
    float* p = at0 + c * step;
    ask(at0 + min(c + 1, count - 1) * step, two);
    work_chunk(p, one);
    if (c + 1 < count) {
      ask(at0 + min(c + 2, count - 1) * step, one);
      work_chunk(p + step, two);
    }
  }
  if (owns) {
#pragma unroll
    for (int t = 0; t < TS; ++t) *reinterpret_cast<f32x4*>(sp + row[t]) = st[t];
  }
}

// O^T = S^T (diag(G) Q)^T + U^T P^T: a lane ends up with four consecutive columns of a row.  A wavefront takes sixteen columns,
// a workgroup 64 of a (chunk, head): with 32 a wavefront two workgroups filled a compute unit's registers (and spilled), 528
// of 128 columns needed a second turn for their last 16, and heads of 64 columns kept two of four wavefronts idle.  33 chunks of 16
// heads of 128 x 128: 24.7 us (38.8); 32 of 32 of 64 x 64 (the generalized rule): 18.2 (32.8).
template <int DIM, bool MORE>
__global__ void __launch_bounds__(DC_THREADS, 3)
delta_chunks_result_kernel(const float* work, const int32_t* __restrict__ chunk_row0,
                           const int32_t* __restrict__ chunk_rows, float* __restrict__ out, int heads, int vdim) {
  constexpr int LD = DIM + 4, LP = DC_ROWS + 4;
  __shared__ __attribute__((aligned(16))) float q_s[DC_ROWS * LD];
  __shared__ __attribute__((aligned(16))) float p_s[DC_ROWS * LP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int head = blockIdx.x, chunk = blockIdx.y;
  const int64_t row0 = chunk_row0[chunk];
  const int n = chunk_rows[chunk];
  const DeltaBlock blk{DIM, vdim, MORE};
  const float* mine = work + (static_cast<int64_t>(chunk) * heads + head) * blk.size();
  // Everything is asked for before the first of it is used (`work` is a plain pointer: loads through a `const __restrict__`
  // one were moved behind the barrier); this wavefront's columns of S and U last, they arrive over the barrier (a tile past
  // the last one: that one, not stored)
  constexpr int NQ = DC_ROWS * DIM / 4 / DC_THREADS, NPP = DC_ROWS * 16 / DC_THREADS;
  const int tile = 4 * blockIdx.z + wave, col0 = 16 * min(tile, vdim / 16 - 1);
  f32x4 qr[NQ], pr[NPP], sa[DIM / 16], ua[4];
#pragma unroll
  for (int i = 0; i < NQ; ++i) qr[i] = *reinterpret_cast<const f32x4*>(mine + blk.q() + 4 * (tid + DC_THREADS * i));
#pragma unroll
  for (int i = 0; i < NPP; ++i) pr[i] = *reinterpret_cast<const f32x4*>(mine + blk.p() + 4 * (tid + DC_THREADS * i));
#pragma unroll
  for (int c = 0; c < DIM / 16; ++c)
    sa[c] = *reinterpret_cast<const f32x4*>(mine + blk.s() + static_cast<int64_t>(col0 + m) * DIM + 16 * c + 4 * g);
#pragma unroll
  for (int s = 0; s < 4; ++s) ua[s] = *reinterpret_cast<const f32x4*>(mine + blk.u() + (col0 + m) * 64 + 16 * s + 4 * g);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int id = tid + DC_THREADS * i;
    *reinterpret_cast<f32x4*>(q_s + id / (DIM / 4) * LD + 4 * (id % (DIM / 4))) = qr[i];
  }
#pragma unroll
  for (int i = 0; i < NPP; ++i) {  // (tiles above the diagonal hold nothing and are not read below)
    const int id = tid + DC_THREADS * i;
    *reinterpret_cast<f32x4*>(p_s + (id >> 4) * LP + 4 * (id & 15)) = pr[i];
  }
  __syncthreads();
  if (16 * tile >= vdim) return;
  const f32x4 none = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 acc[4];  // [tile of rows]
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] = none;
#pragma unroll
  for (int c = 0; c < DIM / 16; ++c) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      acc[r] += dc_mac(sa[c], *reinterpret_cast<const f32x4*>(q_s + (16 * r + m) * LD + 16 * c + 4 * g), none);
    // (added up here: the optimiser would move the sums behind the branches below and keep every addend until then)
#pragma unroll
    for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(acc[r]));
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const bool odd = __any(dc_odd(ua[s]));
#pragma unroll
    for (int r = s; r < 4; ++r) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(p_s + (16 * r + m) * LP + 16 * s + 4 * g);
      if (r == s && odd) acc[r] += dc_mac_block_second(ua[s], b, dc_seen(m, 4 * g, true), none);
      else acc[r] += dc_mac(ua[s], b, none);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 16 * r + m;
    if (row < n) {
      f32x4* to = reinterpret_cast<f32x4*>(out + ((row0 + row) * heads + head) * vdim + 16 * tile + 4 * g);
      if constexpr (MORE) *to += acc[r];  // (Q V is there already)
      else *to = acc[r];
    }
  }
}

// q, k, v, ab, a_log, dt_bias, state, out as ix_delta_rule takes them (bfloat16, a decay per head).  chunk_row0 /
// chunk_rows [chunks]: first row in the step and number of rows (1 to 64) of every chunk; request seq_ids[s] of the
// step has the chunks seq_first[s] .. + seq_count[s], in order; its state is read before them and written after them.
// work: chunks * heads blocks as `DeltaBlock` has them (work_floats: how many floats there are).
extern "C" int ix_delta_chunks(const void* q, const void* k, const void* v, int64_t q_stride, int64_t k_stride,
                               int64_t v_stride, const float* ab, const float* a_log, const float* dt_bias, float* state,
                               int64_t state_stride, const int32_t* state_slots, const int32_t* chunk_row0,
                               const int32_t* chunk_rows, int chunks, const int32_t* seq_ids, const int32_t* seq_first,
                               const int32_t* seq_count, int seqs, float* work, int64_t work_floats, float* out,
                               int heads, int kv_heads, int dim, int vdim, hipStream_t stream) {
  IX_REQUIRE(chunks >= 0 && seqs >= 0 && heads > 0 && kv_heads > 0 && vdim > 0, "sizes must be positive");
  IX_REQUIRE(heads % kv_heads == 0, "heads must be a multiple of kv_heads");
  IX_REQUIRE(dim == 32 || dim == 64 || dim == 128, "key heads of 32, 64 or 128 numbers");
  IX_REQUIRE(vdim % 16 == 0, "value heads in multiples of 16 numbers");
  IX_REQUIRE(state_stride >= static_cast<int64_t>(heads) * dim * vdim && state_stride % 4 == 0, "state blocks too small");
  IX_REQUIRE(q_stride % 8 == 0 && k_stride % 8 == 0, "rows must lie on 16-byte boundaries");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(state) |
               reinterpret_cast<uintptr_t>(work) | reinterpret_cast<uintptr_t>(out)) & 15) == 0,
             "operands must lie on 16-byte boundaries");
  IX_REQUIRE(heads < 65536 && chunks < 65536 && seqs < 65536 && vdim / 16 < 65536, "too many heads, chunks or requests");
  IX_REQUIRE(work_floats >= static_cast<int64_t>(chunks) * heads * (DeltaBlock{dim, vdim, 0}).size(), "workspace too small");
  if (chunks == 0 || seqs == 0) return 0;
#define RUN(DIM)                                                                                                         \
  hipLaunchKernelGGL(delta_chunks_prepare_kernel<DIM>, dim3(heads, chunks), dim3(DC_THREADS), 0, stream, (const bf16_t*)q, \
                     (const bf16_t*)k, (const bf16_t*)v, q_stride, k_stride, v_stride, ab, a_log, dt_bias, chunk_row0,   \
                     chunk_rows, work, heads, kv_heads, vdim);                                                           \
  if (ix_check_launch("ix_delta_chunks: prepare")) return 1;                                                             \
  hipLaunchKernelGGL((delta_chunks_chain_kernel<DIM, false>), dim3(heads, vdim / 16, seqs), dim3(DC_THREADS), 0, stream, work, \
                     seq_ids, seq_first, seq_count, state_slots, state, state_stride, heads, vdim);                      \
  if (ix_check_launch("ix_delta_chunks: chain")) return 1;                                                               \
  hipLaunchKernelGGL((delta_chunks_result_kernel<DIM, false>), dim3(heads, chunks, (vdim + 63) / 64), dim3(DC_THREADS), 0, stream, work, chunk_row0, \
                     chunk_rows, out, heads, vdim)
  if (dim == 32) { RUN(32); }
  else if (dim == 64) { RUN(64); }
  else { RUN(128); }
#undef RUN
  return ix_check_launch("ix_delta_chunks");
}

// The generalized rule: r, k [T, heads * dim] and v [T, heads * vdim] bfloat16 rows, w, a, b float32 [T, heads * dim] as
// ix_linear_state takes them (every decay between e^-1 and 1); the rest as above, blocks of the workspace with `m`.
extern "C" int ix_general_delta_chunks(const void* r, const void* k, const void* v, int64_t r_stride, int64_t k_stride,
                                       int64_t v_stride, const float* w_rows, const float* a_rows, const float* b_rows,
                                       float* state, int64_t state_stride, const int32_t* state_slots,
                                       const int32_t* chunk_row0, const int32_t* chunk_rows, int chunks,
                                       const int32_t* seq_ids, const int32_t* seq_first, const int32_t* seq_count, int seqs,
                                       float* work, int64_t work_floats, float* out, int heads, int dim, int vdim,
                                       hipStream_t stream) {
  IX_REQUIRE(chunks >= 0 && seqs >= 0 && heads > 0 && vdim > 0, "sizes must be positive");
  IX_REQUIRE(dim == 32 || dim == 64 || dim == 128, "key heads of 32, 64 or 128 numbers");
  IX_REQUIRE(vdim % 16 == 0, "value heads in multiples of 16 numbers");
  IX_REQUIRE(state_stride >= static_cast<int64_t>(heads) * dim * vdim && state_stride % 4 == 0, "state blocks too small");
  IX_REQUIRE(((reinterpret_cast<uintptr_t>(state) | reinterpret_cast<uintptr_t>(work) | reinterpret_cast<uintptr_t>(out)) & 15) == 0,
             "state, workspace and result must lie on 16-byte boundaries");
  IX_REQUIRE(heads < 65536 && chunks < 65536 && seqs < 65536 && vdim / 16 < 65536, "too many heads, chunks or requests");
  IX_REQUIRE(work_floats >= static_cast<int64_t>(chunks) * heads * (DeltaBlock{dim, vdim, 1}).size(), "workspace too small");
  if (chunks == 0 || seqs == 0) return 0;
#define RUN(DIM)                                                                                                         \
  hipLaunchKernelGGL(general_chunks_prepare_kernel<DIM>, dim3(heads, chunks), dim3(DC_THREADS), 0, stream,               \
                     (const bf16_t*)r, (const bf16_t*)k, (const bf16_t*)v, r_stride, k_stride, v_stride, w_rows, a_rows, \
                     b_rows, chunk_row0, chunk_rows, work, out, heads, vdim);                                            \
  if (ix_check_launch("ix_general_delta_chunks: prepare")) return 1;                                                     \
  hipLaunchKernelGGL((delta_chunks_chain_kernel<DIM, true>), dim3(heads, vdim / 16, seqs), dim3(DC_THREADS), 0, stream,  \
                     work, seq_ids, seq_first, seq_count, state_slots, state, state_stride, heads, vdim);                \
  if (ix_check_launch("ix_general_delta_chunks: chain")) return 1;                                                       \
  hipLaunchKernelGGL((delta_chunks_result_kernel<DIM, true>), dim3(heads, chunks, (vdim + 63) / 64), dim3(DC_THREADS), 0, stream, work,    \
                     chunk_row0, chunk_rows, out, heads, vdim)
  if (dim == 32) { RUN(32); }
  else if (dim == 64) { RUN(64); }
  else { RUN(128); }
#undef RUN
  return ix_check_launch("ix_general_delta_chunks");
}
