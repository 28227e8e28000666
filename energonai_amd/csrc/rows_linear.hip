// Projections of a few rows (the newest token of up to 32 sequences), and the decode step of a pre-LN block on top of
// them: five launches instead of the eleven of LayerNorm, library GEMM, K/V append, length update, attention, GEMM,
// residual + LayerNorm, GEMM with activation, GEMM, residual add, history copy.
//
//   y = act(LayerNorm(x) W^T + b) (+ residual)         x [R,K], W [N,K] (torch.nn.Linear's layout), R <= 32
//
// What bounds it: for narrow models the chain launch -> first weight bytes -> last MFMA -> store, for wide ones the bytes of
// the weights.  So a workgroup takes few output columns (eight or sixteen a tile) and its waves split K between them, 64 or
// 128 channels a step: every lane's weight loads of the first steps are sent for before anything is waited for, each wave
// needs few steps, and the partial sums meet once, in LDS.  W rows are the A operand of the 16x16x32 MFMA (lane j of 16 holds
// row n0 + j, 32 bytes = 16 channels of it per step: the four lane groups together 128 contiguous bytes a row), the x rows
// the B operand with the same channel order, so the result leaves each lane with four consecutive columns of one row.
//
// The LayerNorm in front of a projection is computed where its result is consumed: the B fragments of all waves together
// are the rows, so mean and centred squares (fp32) come from registers, and each fragment is normalised and rounded to the
// storage type, exactly what a LayerNorm kernel would have stored.  That takes rows that fit: up to kMaxWidth channels.
#include "common.hip.h"

#include <math.h>

#include <type_traits>

namespace en {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kMaxWidth = EN_BLOCK_DECODE_MAX_HIDDEN;
constexpr int kMaxRows = EN_BLOCK_DECODE_MAX_BATCH;

enum RowsIn { kPlain, kNorm16, kNormF32 };                 // 16-bit rows; LayerNorm of 16-bit rows; LayerNorm of fp32 rows
enum RowsOut { kStore, kResidualF32, kAddF32, kScatterKVQ };   // see RowsArgs

struct RowsArgs {
  const void *x;              // [R] rows of K, x_stride elements apart
  int64_t x_stride;
  int R, K, N;
  const void *w, *bias;       // [N,K]; [N] or null
  const void *gamma, *beta;   // LayerNorm in front
  float eps;
  int act;                    // EN_ACT_*
  void *y;                    // kStore: 16-bit; kResidualF32: fp32, sum with 16-bit `res`; kAddF32: 16-bit, sum with fp32 `res`
  int64_t y_stride;
  const void *res;
  int64_t res_stride;
  int32_t *advance;           // if set, `advance[r]` of every row goes up by one: lengths that nobody reads any more in this launch
  // kScatterKVQ: N = 3 hidden columns ordered k, v, q.  K and V go to position kv_lens[r] of their caches, q to y.
  void *k_cache, *v_cache;
  const int32_t *kv_lens;
  int hidden, D, Sk;
  int64_t c_sb, c_sh, c_ss;
  const int32_t *page_table;  // paged caches: c_sb is the page stride
  int max_pages, lg_page, num_pages;
};

template <int DT>
__device__ __forceinline__ floatx4 mfma16(const uint4 &a, const uint4 &b, floatx4 c) {
  if constexpr (DT == EN_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ float activate(float v, int act) {
  switch (act) {
    case EN_ACT_RELU: return v < 0.f ? 0.f : v;      // NaN stays NaN
    case EN_ACT_GELU_TANH: return 0.5f * v * (1.f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
    case EN_ACT_GELU: return 0.5f * v * (1.f + erff(v * 0.7071067811865476f));
    default: return v;
  }
}

// RT: row tiles.  1, 2: sixteen rows each, sixteen columns per column tile, a step is 64 channels.  0: up to eight rows.  The
// MFMA's sixteen A rows are then eight columns at the lower and the same eight at the upper half of a step of 128 channels,
// its sixteen B columns the eight rows at those halves; the two quadrants where the halves meet are the result and the other
// two are dropped.  No lane loads a row that is not there, and a column tile of eight makes twice the workgroups.
// CT: column tiles per workgroup.
template <int DT, int IN, int OUT, int NW, int U, int RT, int CT>
__global__ __launch_bounds__(NW * kWave) void rows_linear_kernel(RowsArgs a) {
  typedef Elem<DT> E;
  typedef typename E::T T;
  typedef Pack<T, 8> P8;
  constexpr bool HALF = RT == 0;
  constexpr int RTILES = HALF ? 1 : RT;
  constexpr int ROWS = HALF ? 8 : 16;           // rows per row tile, columns per column tile
  constexpr int BK = HALF ? 128 : 64;           // channels per wave and step: two MFMAs per tile
  constexpr int XV = IN == kNormF32 ? 4 : 2;    // 16-byte loads of 16 channels of a row
  constexpr bool NORM = IN != kPlain;
  static_assert(RTILES * CT < NW && kMaxRows <= kWave, "a wave is left to move the lengths on");
  __shared__ __attribute__((aligned(16))) float s_acc[NW][RTILES * CT][kWave][4];
  __shared__ float s_sum[NORM ? 2 : 1][NW][RTILES * 16];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int j = lane & 15, g = lane >> 4;
  const int jr = HALF ? (j & 7) : j;            // row of the tile and column of the tile that this lane loads
  const int kl = (HALF ? (j >> 3) * 64 : 0) + g * 16;   // its 16 channels of a step
  const int n0 = blockIdx.x * ROWS * CT;
  const int nsteps = (a.K + BK - 1) / BK;

  // Bounds-checked buffer loads: columns past N, rows past R, channels past K and steps past the end arrive as zeros without
  // a branch (branches around the loads, each with its own wait, cost a factor of 2.5).
  constexpr int XS = IN == kNormF32 ? 4 : 2;
  const rsrc_t w_rsrc = make_rsrc(reinterpret_cast<const T *>(a.w) + (int64_t)n0 * a.K, (uint32_t)min(ROWS * CT, a.N - n0) * (uint32_t)a.K * 2u);
  const rsrc_t x_rsrc = make_rsrc(a.x, (uint32_t)(((int64_t)(a.R - 1) * a.x_stride + a.K) * XS));
  const rsrc_t g_rsrc = make_rsrc(a.gamma, NORM ? (uint32_t)a.K * 2u : 0u), b_rsrc = make_rsrc(a.beta, NORM ? (uint32_t)a.K * 2u : 0u);
  uint32_t xrow[RTILES];
#pragma unroll
  for (int t = 0; t < RTILES; ++t) xrow[t] = t * 16 + jr < a.R ? (uint32_t)((int64_t)(t * 16 + jr) * a.x_stride * XS) : kOutOfRange;

  // In front of a LayerNorm the rows go out ahead of the weights, with gamma and beta of the wave's steps: loads complete in
  // order, and the statistics then run while the weights travel.  What the end needs is sent for here too.  (Two row tiles on
  // sixteen waves have no registers for any of it.)  768 -> 2304 with LayerNorm, 8 rows, 5.9 -> 4.8 us, 768 -> 3072 5.5 -> 4.7; a
  // block's five launches of a step 22.7 -> 21.6 us, 8 rows of 1024 30.2 -> 28.1, 16 of 2048 55.8 -> 53.6.
  constexpr bool AHEAD = !(NORM && NW == 16 && RTILES == 2);
  uint4 w[U][CT][2], x[U][RTILES][XV], ga[U][2], be[U][2];
  enum { kW = 1, kX = 2 };
  auto fetch = [&](auto what, int u, int step) {
    const int k = step * BK + kl;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const uint32_t in = k + 8 * half < a.K ? 0u : kOutOfRange;
      if constexpr (decltype(what)::value & kW)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          w[u][c][half] = buffer_load16(w_rsrc, ((uint32_t)(c * ROWS + jr) * (uint32_t)a.K + (uint32_t)(k + 8 * half)) * 2u | in);
      if constexpr (decltype(what)::value & kX)
#pragma unroll
        for (int t = 0; t < RTILES; ++t)
#pragma unroll
          for (int v = 0; v < XV / 2; ++v)
            x[u][t][half * (XV / 2) + v] = buffer_load16(x_rsrc, xrow[t] + (uint32_t)(k + 8 * half) * XS + v * 16 | xrow[t] & kOutOfRange | in);
    }
  };
  const std::integral_constant<int, kW> weights;
  const std::integral_constant<int, kX> rows;
  const std::integral_constant<int, kW | kX> both;
  auto load_affine = [&](int u, int half, int k) {
    ga[u][half] = buffer_load16(g_rsrc, (uint32_t)(k + 8 * half) * 2u);
    be[u][half] = buffer_load16(b_rsrc, (uint32_t)(k + 8 * half) * 2u);
  };
  if constexpr (AHEAD)
#pragma unroll
    for (int u = 0; u < U; ++u) fetch(rows, u, wave + u * NW);
  if constexpr (NORM && AHEAD)
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int half = 0; half < 2; ++half) load_affine(u, half, (wave + u * NW) * BK + kl);

  // What the waves that finish a tile need besides the sums is sent for here too: behind them it would be another trip to
  // memory.  Wave t CT + c finishes row tile t of column tile c: lane (j, g) has columns 4g .. 4g + 3 of row j; with eight rows
  // lanes (j, g) and (j + 8, g + 2) hold the halves of columns 4g .. of row j, j < 8, g < 2.
  typedef Pack<T, 4> P4;
  typedef Pack<float, 4> F4;
  const int r = wave / CT * 16 + j, n = n0 + wave % CT * ROWS + 4 * g;
  const bool finishes = wave < RTILES * CT && r < a.R && n < a.N && !(HALF && (j >= 8 || g >= 2));
  P4 bias4{}, res4{};
  F4 add4{};
  int pos = 0;
  auto load_finish = [&] {
    if (!finishes) return;
    if (a.bias) bias4 = load_pack<T, 4>(reinterpret_cast<const T *>(a.bias) + n);
    if constexpr (OUT == kResidualF32) res4 = load_pack<T, 4>(reinterpret_cast<const T *>(a.res) + r * a.res_stride + n);
    if constexpr (OUT == kAddF32) add4 = load_pack<float, 4>(reinterpret_cast<const float *>(a.res) + r * a.res_stride + n);
    if constexpr (OUT == kScatterKVQ) pos = a.kv_lens[r];
  };
  if constexpr (AHEAD) load_finish();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if constexpr (AHEAD) fetch(weights, u, wave + u * NW);
    else fetch(both, u, wave + u * NW);
  }

  // element e of the 16 channels that this lane holds of row tile t in step u
  auto x_at = [&](int u, int t, int e) {
    if constexpr (IN == kNormF32) return __builtin_bit_cast(Pack<float, 4>, x[u][t][e / 4]).v[e % 4];
    else return E::to_float(__builtin_bit_cast(P8, x[u][t][e / 8]).v[e % 8]);
  };
  float mu[RTILES], inv[RTILES];
  if constexpr (NORM) {
    // The U steps of the NW waves are the whole row (the host sees to it): mean and centred squares come from the fragments
    // in registers, over the lane groups by permlane swaps and over the waves through LDS.
    auto row_sum = [&](float (&v)[RTILES], float (&slots)[NW][RTILES * 16]) {
#pragma unroll
      for (int t = 0; t < RTILES; ++t) {
        float f = v[t];
        if constexpr (HALF) f += dpp_move<0x128>(f);        // row_ror:8, the other half of the step
        auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(f), __float_as_uint(f), false, false);
        f = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        r = __builtin_amdgcn_permlane32_swap(__float_as_uint(f), __float_as_uint(f), false, false);
        f = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        if (g == 0) slots[wave][t * 16 + j] = f;
      }
      lds_barrier();
#pragma unroll
      for (int t = 0; t < RTILES; ++t) {
        v[t] = 0.f;
#pragma unroll
        for (int k = 0; k < NW; ++k) v[t] += slots[k][t * 16 + j];
      }
    };
    float s[RTILES], d2[RTILES];
#pragma unroll
    for (int t = 0; t < RTILES; ++t) {
      s[t] = 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[t] += x_at(u, t, e);      // channels past K are zeros
    }
    row_sum(s, s_sum[0]);
#pragma unroll
    for (int t = 0; t < RTILES; ++t) {
      mu[t] = s[t] / (float)a.K;
      d2[t] = 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int half = 0; half < 2; ++half)
          if ((wave + u * NW) * BK + kl + 8 * half < a.K) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float d = x_at(u, t, 8 * half + e) - mu[t];
              d2[t] += d * d;
            }
          }
    }
    row_sum(d2, s_sum[NORM ? 1 : 0]);
#pragma unroll
    for (int t = 0; t < RTILES; ++t) inv[t] = 1.0f / sqrtf(d2[t] / (float)a.K + a.eps);
  }

  floatx4 acc[RTILES][CT];
#pragma unroll
  for (int t = 0; t < RTILES; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[t][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = wave; s0 < nsteps; s0 += NW * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        if constexpr (NORM && !AHEAD) load_affine(u, half, (s0 + u * NW) * BK + kl);
#pragma unroll
        for (int t = 0; t < RTILES; ++t) {
          uint4 b;
          if constexpr (NORM) {
            const P8 gp = __builtin_bit_cast(P8, ga[u][half]), bp = __builtin_bit_cast(P8, be[u][half]);
            P8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e)
              o.v[e] = E::from_float((x_at(u, t, half * 8 + e) - mu[t]) * inv[t] * E::to_float(gp.v[e]) + E::to_float(bp.v[e]));
            b = __builtin_bit_cast(uint4, o);
          } else {
            b = x[u][t][half];
          }
#pragma unroll
          for (int c = 0; c < CT; ++c) acc[t][c] = mfma16<DT>(w[u][c][half], b, acc[t][c]);
        }
      }
      if constexpr (!NORM) fetch(both, u, s0 + (u + U) * NW);
    }
  }

#pragma unroll
  for (int t = 0; t < RTILES; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) *reinterpret_cast<floatx4 *>(s_acc[wave][t * CT + c][lane]) = acc[t][c];
  lds_barrier();
  // by a wave that finishes no tile
  if (a.advance && blockIdx.x == 0 && wave == NW - 1 && lane < a.R) a.advance[lane] += 1;
  if constexpr (!AHEAD) load_finish();
  if (!finishes) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < NW; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] += s_acc[k][wave][lane][i];
      if constexpr (HALF) v[i] += s_acc[k][wave][(lane + 40) % kWave][i];
    }
  if (a.bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += E::to_float(bias4.v[i]);
  }
  P4 o;
  if constexpr (OUT == kStore) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = E::from_float(activate(v[i], a.act));
    store_pack<T, 4>(reinterpret_cast<T *>(a.y) + r * a.y_stride + n, o);
  } else if constexpr (OUT == kResidualF32) {
    F4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) f.v[i] = v[i] + E::to_float(res4.v[i]);
    store_pack<float, 4>(reinterpret_cast<float *>(a.y) + r * a.y_stride + n, f);
  } else if constexpr (OUT == kAddF32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = E::from_float(v[i] + add4.v[i]);
    store_pack<T, 4>(reinterpret_cast<T *>(a.y) + r * a.y_stride + n, o);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = E::from_float(v[i]);
    const int part = n / a.hidden, c = n - part * a.hidden;
    if (part == 2) {
      store_pack<T, 4>(reinterpret_cast<T *>(a.y) + r * a.y_stride + c, o);
      return;
    }
    const int h = c / a.D, d = c - h * a.D;
    int64_t at = (int64_t)r * a.c_sb + (int64_t)pos * a.c_ss;
    bool room = pos >= 0 && pos < a.Sk;
    if (a.page_table) {
      const int pi = pos >> a.lg_page;
      const int id = (room && pi < a.max_pages) ? a.page_table[(int64_t)r * a.max_pages + pi] : -1;
      room = (unsigned)id < (unsigned)a.num_pages;
      at = (int64_t)id * a.c_sb + (int64_t)(pos & ((1 << a.lg_page) - 1)) * a.c_ss;
    }
    if (room) store_pack<T, 4>(reinterpret_cast<T *>(part == 0 ? a.k_cache : a.v_cache) + at + (int64_t)h * a.c_sh + d, o);
  }
}

template <int DT, int IN, int OUT, int NW, int U, int RT, int CT = 1>
static int launch_rows_linear(const RowsArgs &a, hipStream_t s) {
  constexpr int COLS = (RT == 0 ? 8 : 16) * CT;
  rows_linear_kernel<DT, IN, OUT, NW, U, RT, CT><<<(unsigned)ceil_div(a.N, COLS), NW * kWave, 0, s>>>(a);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

// Waves per workgroup, steps in flight per wave, row tiles and column tiles, by the rows R and the width K.  With a LayerNorm
// in front the waves and steps have to hold the whole row, and its arithmetic is shared by more columns.  Measured alone with
// cold weights (launch to launch, 2.8 us of it an empty launch; the library's GEMM, without LayerNorm, in brackets), 8 rows:
//   768 -> 768   3 x 2 steps 2.9 us, 6 x 1 3.1, sixteen rows' tile 4 x 3 3.3 (4.0)
//   3072 -> 768  8 x 3 5.6 us, 12 x 2 5.8, sixteen rows' tile 16 x 3 7.8 (5.4);      8192 -> 2048 10.7 us, 15.7 (9.6)
//   768 -> 2304 with LayerNorm 6 x 1, two column tiles 4.1 us, one 4.6, sixteen rows' tile 4.5 (4.0 + a LayerNorm)
//   2048 -> 6144 with LayerNorm 8 x 2, four column tiles 7.8 us, two 9.5, one 10.2 (8.9 + a LayerNorm)
// 16 rows 2048 -> 6144 with LayerNorm: two column tiles 9.7 us, one 14.9; 24 rows: 14.0, 20.6.
template <int DT, int IN, int OUT>
static int rows_linear(const RowsArgs &a, hipStream_t s) {
  const int64_t steps = ceil_div(a.K, 64), wide = ceil_div(a.K, 128);
  if constexpr (IN == kPlain) {
    if (a.R <= 8) {
      if (wide <= 6) return launch_rows_linear<DT, IN, OUT, 3, 2, 0, 1>(a, s);
      if (wide <= 16) return launch_rows_linear<DT, IN, OUT, 8, 2, 0, 1>(a, s);
      return launch_rows_linear<DT, IN, OUT, 8, 3, 0, 1>(a, s);
    }
    if (a.R <= 16) {
      if (steps <= 16) return launch_rows_linear<DT, IN, OUT, 4, 3, 1, 1>(a, s);
      if (steps <= 32) return launch_rows_linear<DT, IN, OUT, 8, 3, 1, 1>(a, s);
      return launch_rows_linear<DT, IN, OUT, 16, 3, 1, 1>(a, s);
    }
    if (steps <= 16) return launch_rows_linear<DT, IN, OUT, 4, 2, 2, 1>(a, s);
    if (steps <= 32) return launch_rows_linear<DT, IN, OUT, 8, 2, 2, 1>(a, s);
    return launch_rows_linear<DT, IN, OUT, 16, 2, 2, 1>(a, s);
  } else {
    if (steps > 32) return EN_ERR_UNSUPPORTED;
    if (a.R <= 8) {
      if (wide <= 6) return launch_rows_linear<DT, IN, OUT, 6, 1, 0, 2>(a, s);
      if (a.N < 4096) return launch_rows_linear<DT, IN, OUT, 8, 2, 0, 2>(a, s);
      return launch_rows_linear<DT, IN, OUT, 8, 2, 0, 4>(a, s);
    }
    if (a.R <= 16) {
      if (steps <= 12) return launch_rows_linear<DT, IN, OUT, 4, 3, 1, 2>(a, s);
      if (steps <= 24) return launch_rows_linear<DT, IN, OUT, 8, 3, 1, 2>(a, s);
      return launch_rows_linear<DT, IN, OUT, 16, 2, 1, 2>(a, s);
    }
    if (steps <= 16) return launch_rows_linear<DT, IN, OUT, 8, 2, 2, 2>(a, s);
    return launch_rows_linear<DT, IN, OUT, 16, 2, 2, 2>(a, s);
  }
}

static int log2_page(int v) {
  int lg = 0;
  while ((1 << lg) < v) ++lg;
  return (1 << lg) == v ? lg : -1;
}

template <int DT>
static int block_decode(const en_block_decode_args &p, hipStream_t s) {
  const int64_t hid = (int64_t)p.head_num * p.size_per_head;
  const int R = p.batch;
  unsigned char *ws = static_cast<unsigned char *>(p.workspace);
  auto take = [&](int64_t bytes) {
    unsigned char *at = ws;
    ws += (bytes + 255) / 256 * 256;
    return at;
  };
  void *q = take(R * hid * 2), *ctx = take(R * hid * 2), *sum = take(R * hid * 4), *h = take(R * p.mlp_width * 2);
  const int64_t attn_bytes = en_decode_attn_workspace_bytes(R, p.head_num, p.cache_len, p.size_per_head);
  void *attn_ws = take(attn_bytes);
  auto attend = [&](bool launch) {
    return decode_attn_ahead(q, p.k_cache, p.v_cache, ctx, p.kv_lens, p.page_table, R, p.head_num, p.cache_len, p.max_pages_per_seq,
                             p.page_size, p.num_pages, p.size_per_head, p.cache_strides, p.scale, p.dtype, attn_ws, attn_bytes, launch, s);
  };
  int rc = attend(false);      // whatever the attention refuses, before the caches are written
  if (rc) return rc;

  // k, v, q of the new tokens; K and V straight into the caches
  RowsArgs a{};
  a.x = p.x; a.x_stride = p.x_stride; a.R = R; a.K = (int)hid; a.N = (int)(3 * hid);
  a.w = p.qkv_weight; a.bias = p.qkv_bias; a.gamma = p.norm1_weight; a.beta = p.norm1_bias; a.eps = p.norm1_eps;
  a.y = q; a.y_stride = hid;
  a.k_cache = p.k_cache; a.v_cache = p.v_cache; a.kv_lens = p.kv_lens; a.hidden = (int)hid; a.D = p.size_per_head; a.Sk = p.cache_len;
  a.c_sb = p.cache_strides[0]; a.c_sh = p.cache_strides[1]; a.c_ss = p.cache_strides[2];
  a.page_table = p.page_table; a.max_pages = p.max_pages_per_seq; a.num_pages = p.num_pages;
  a.lg_page = p.page_table ? log2_page(p.page_size) : 0;
  rc = rows_linear<DT, kNorm16, kScatterKVQ>(a, s);
  if (rc) return rc;
  // attention over the caches, the new position included
  rc = attend(true);
  if (rc) return rc;
  // output projection + residual; the lengths move on behind the last kernel that reads the old ones
  RowsArgs d{};
  d.x = ctx; d.x_stride = hid; d.R = R; d.K = (int)hid; d.N = (int)hid; d.w = p.dense_weight; d.bias = p.dense_bias;
  d.y = sum; d.y_stride = hid; d.res = p.x; d.res_stride = p.x_stride; d.advance = p.kv_lens;
  rc = rows_linear<DT, kPlain, kResidualF32>(d, s);
  if (rc) return rc;
  // MLP on the normalised sum, added to the sum
  RowsArgs m{};
  m.x = sum; m.x_stride = hid; m.R = R; m.K = (int)hid; m.N = (int)p.mlp_width; m.w = p.mlp1_weight; m.bias = p.mlp1_bias;
  m.gamma = p.norm2_weight; m.beta = p.norm2_bias; m.eps = p.norm2_eps; m.act = p.activation; m.y = h; m.y_stride = p.mlp_width;
  rc = rows_linear<DT, kNormF32, kStore>(m, s);
  if (rc) return rc;
  RowsArgs f{};
  f.x = h; f.x_stride = p.mlp_width; f.R = R; f.K = (int)p.mlp_width; f.N = (int)hid; f.w = p.mlp2_weight; f.bias = p.mlp2_bias;
  f.y = p.y; f.y_stride = p.y_stride; f.res = sum; f.res_stride = hid;
  return rows_linear<DT, kPlain, kAddF32>(f, s);
}

}  // namespace en

extern "C" {

int64_t en_block_decode_workspace_bytes(int batch, int head_num, int size_per_head, int64_t mlp_width, int cache_len) {
  if (batch < 1 || head_num < 1 || size_per_head < 1 || mlp_width < 1 || cache_len < 1) return 0;
  const int64_t hid = (int64_t)head_num * size_per_head;
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  return 2 * up(batch * hid * 2) + up(batch * hid * 4) + up(batch * mlp_width * 2) +
         up(en_decode_attn_workspace_bytes(batch, head_num, cache_len, size_per_head));
}

int en_block_decode(const en_block_decode_args *p, en_stream_t stream) {
  using namespace en;
  if (!p) return EN_ERR_NULL;
  if (!p->x || !p->norm1_weight || !p->norm1_bias || !p->qkv_weight || !p->dense_weight || !p->norm2_weight || !p->norm2_bias ||
      !p->mlp1_weight || !p->mlp2_weight || !p->k_cache || !p->v_cache || !p->kv_lens || !p->y || !p->workspace)
    return EN_ERR_NULL;
  if (p->dtype != EN_F16 && p->dtype != EN_BF16) return EN_ERR_DTYPE;
  if (p->batch < 1 || p->head_num < 1 || p->size_per_head < 1 || p->mlp_width < 1 || p->cache_len < 1) return EN_ERR_SHAPE;
  const int64_t hid = (int64_t)p->head_num * p->size_per_head;
  // the kernel's offsets into kMaxRows rows of the MLP's width and into sixteen columns of its weights are 32-bit bytes, the sign bit marking "absent"
  if (p->batch > kMaxRows || hid > kMaxWidth || p->size_per_head % 8 || p->size_per_head > 512 || p->mlp_width % 8 ||
      p->mlp_width * kMaxRows * 2 >= (1ll << 31))
    return EN_ERR_UNSUPPORTED;
  if ((int64_t)p->batch * p->x_stride * 2 >= (1ll << 31) || p->activation < EN_ACT_NONE || p->activation > EN_ACT_GELU) return EN_ERR_UNSUPPORTED;
  if (p->page_table && (log2_page(p->page_size) < 4 || p->max_pages_per_seq < 1 || p->num_pages < 1)) return EN_ERR_UNSUPPORTED;
  if (p->workspace_bytes < en_block_decode_workspace_bytes(p->batch, p->head_num, p->size_per_head, p->mlp_width, p->cache_len))
    return EN_ERR_SCRATCH;
  for (const void *v : {p->x, p->norm1_weight, p->norm1_bias, p->qkv_weight, p->dense_weight, p->norm2_weight, p->norm2_bias,
                        p->mlp1_weight, p->mlp2_weight, (const void *)p->k_cache, (const void *)p->v_cache, (const void *)p->workspace})
    if (!aligned_to(v, 16)) return EN_ERR_ALIGN;
  for (const void *v : {p->qkv_bias, p->dense_bias, p->mlp1_bias, p->mlp2_bias, (const void *)p->y})
    if (v && !aligned_to(v, 8)) return EN_ERR_ALIGN;
  if (p->x_stride % 8 || p->y_stride % 4 || p->x_stride < hid || p->y_stride < hid) return EN_ERR_ALIGN;
  for (int i = 0; i < 3; ++i)
    if (p->cache_strides[i] < 0 || p->cache_strides[i] % 8) return EN_ERR_ALIGN;
  return p->dtype == EN_F16 ? block_decode<EN_F16>(*p, (hipStream_t)stream) : block_decode<EN_BF16>(*p, (hipStream_t)stream);
}

}  // extern "C"
