// Projections of a few rows (the newest token of up to 32 sequences), and the decode step of a pre-LN block on top of
// them: five launches instead of the eleven of LayerNorm, library GEMM, K/V append, length update, attention, GEMM,
// residual + LayerNorm, GEMM with activation, GEMM, residual add, history copy.
//
//   y = act(LayerNorm(x) W^T + b) (+ residual)         x [R,K], W [N,K] (torch.nn.Linear's layout), R <= 32
//
// What bounds it: for narrow models the chain launch -> first weight bytes -> last MFMA -> store (3.5..5 us a kernel, of
// which 2.8 are an empty launch), for wide ones the weights' bytes.  So a workgroup takes 16 output columns only (N / 16
// workgroups) and its waves split K between them, 64 channels a step: every lane's weight loads of the first steps are
// sent for before anything is waited for, each wave needs few steps (three for K = 768 on four waves), and the partial
// sums meet once, in LDS.  W rows are the A operand of the 16x16x32 MFMA (lane j of 16 holds row n0 + j, 32 bytes = 16
// channels of it per step: the four lane groups together 128 contiguous bytes a row), the x rows the B operand with the
// same channel order, so the result leaves each lane with four consecutive columns of one row.
//
// The LayerNorm in front of a projection is computed where its result is consumed: 16 lanes per row take mean and centred
// squares (two passes, fp32), and the B fragments are normalised and rounded to the storage type as they are loaded,
// exactly what a LayerNorm kernel would have stored.  Every workgroup repeats the statistics, so this is for rows of up to
// kMaxWidth channels.
#include "common.hip.h"

#include <math.h>

namespace en {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kMaxWidth = 2048;
constexpr int kMaxRows = 32;

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
    case EN_ACT_RELU: return fmaxf(v, 0.f);
    case EN_ACT_GELU_TANH: return 0.5f * v * (1.f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
    case EN_ACT_GELU: return 0.5f * v * (1.f + erff(v * 0.7071067811865476f));
    default: return v;
  }
}

template <int DT, int IN, int OUT, int NW, int RT>
__global__ __launch_bounds__(NW * kWave) void rows_linear_kernel(RowsArgs a) {
  typedef Elem<DT> E;
  typedef typename E::T T;
  typedef Pack<T, 8> P8;
  constexpr int BK = 64;                        // channels per wave and step: two MFMAs
  constexpr int U = RT == 1 ? 3 : 2;            // steps in flight
  constexpr int XV = IN == kNormF32 ? 4 : 2;    // 16-byte loads of 16 channels of a row
  constexpr bool NORM = IN != kPlain;
  __shared__ __attribute__((aligned(16))) float s_acc[NW][RT][kWave][4];
  __shared__ float s_mu[RT * 16], s_inv[RT * 16];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int j = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int nsteps = (a.K + BK - 1) / BK;

  const T *wrow = reinterpret_cast<const T *>(a.w) + (int64_t)min(n0 + j, a.N - 1) * a.K;
  const unsigned char *xrow[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
    xrow[t] = reinterpret_cast<const unsigned char *>(a.x) + (int64_t)min(t * 16 + j, a.R - 1) * a.x_stride * (IN == kNormF32 ? 4 : 2);
  const T *gamma = reinterpret_cast<const T *>(a.gamma), *beta = reinterpret_cast<const T *>(a.beta);

  uint4 w[U][2], x[U][RT][XV], ga[NORM ? U : 1][2], be[NORM ? U : 1][2];
  auto fetch = [&](int u, int step) {           // a step past the end, and channels past K, arrive as zeros
    const int k = step * BK + g * 16;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const bool in = k + 8 * half < a.K;
      w[u][half] = in ? load16<false>(wrow + k + 8 * half) : make_uint4(0, 0, 0, 0);
      if constexpr (NORM) {
        ga[u][half] = in ? load16<false>(gamma + k + 8 * half) : make_uint4(0, 0, 0, 0);
        be[u][half] = in ? load16<false>(beta + k + 8 * half) : make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int v = 0; v < XV / 2; ++v)
          x[u][t][half * (XV / 2) + v] = in ? load16<false>(xrow[t] + (int64_t)(k + 8 * half) * (XV / 2) * 2 + v * 16) : make_uint4(0, 0, 0, 0);
    }
  };
#pragma unroll
  for (int u = 0; u < U; ++u) fetch(u, wave + u * NW);

  float mu[RT], inv[RT];
  if constexpr (NORM) {
    constexpr int EX = IN == kNormF32 ? 4 : 8;  // elements per 16-byte vector of a row
    constexpr int UV = 8;                       // vectors in flight per lane
    for (int r = tid / 16; r < a.R; r += NW * 4) {
      const unsigned char *row = reinterpret_cast<const unsigned char *>(a.x) + (int64_t)r * a.x_stride * (16 / EX);
      const int nvec = a.K / EX;
      auto pass = [&](auto &&f) {
        for (int v0 = j; v0 < nvec; v0 += 16 * UV) {
          uint4 q[UV];
#pragma unroll
          for (int i = 0; i < UV; ++i)
            if (v0 + 16 * i < nvec) q[i] = load16<false>(row + (int64_t)(v0 + 16 * i) * 16);
#pragma unroll
          for (int i = 0; i < UV; ++i)
            if (v0 + 16 * i < nvec) {
              if constexpr (IN == kNormF32) {
                const Pack<float, 4> p = __builtin_bit_cast(Pack<float, 4>, q[i]);
#pragma unroll
                for (int e = 0; e < 4; ++e) f(p.v[e]);
              } else {
                const P8 p = __builtin_bit_cast(P8, q[i]);
#pragma unroll
                for (int e = 0; e < 8; ++e) f(E::to_float(p.v[e]));
              }
            }
        }
      };
      float s = 0.f, d2 = 0.f;
      pass([&](float v) { s += v; });
      const float m = group_allreduce<OpSum, 16>(s) / (float)a.K;
      pass([&](float v) { d2 += (v - m) * (v - m); });
      d2 = group_allreduce<OpSum, 16>(d2);
      if (j == 0) { s_mu[r] = m; s_inv[r] = 1.0f / sqrtf(d2 / (float)a.K + a.eps); }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const int r = min(t * 16 + j, a.R - 1);
      mu[t] = s_mu[r];
      inv[t] = s_inv[r];
    }
  }

  floatx4 acc[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = wave; s0 < nsteps; s0 += NW * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          uint4 b;
          if constexpr (NORM) {
            const P8 gp = __builtin_bit_cast(P8, ga[u][half]), bp = __builtin_bit_cast(P8, be[u][half]);
            P8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              float v;
              if constexpr (IN == kNormF32) v = __builtin_bit_cast(Pack<float, 4>, x[u][t][half * 2 + e / 4]).v[e % 4];
              else v = E::to_float(__builtin_bit_cast(P8, x[u][t][half]).v[e]);
              o.v[e] = E::from_float((v - mu[t]) * inv[t] * E::to_float(gp.v[e]) + E::to_float(bp.v[e]));
            }
            b = __builtin_bit_cast(uint4, o);
          } else {
            b = x[u][t][half];
          }
          acc[t] = mfma16<DT>(w[u][half], b, acc[t]);
        }
      fetch(u, s0 + (u + U) * NW);
    }
  }

#pragma unroll
  for (int t = 0; t < RT; ++t) *reinterpret_cast<floatx4 *>(s_acc[wave][t][lane]) = acc[t];
  if (a.advance && blockIdx.x == 0 && tid < a.R) a.advance[tid] += 1;
  __syncthreads();
  if (wave >= RT) return;
  // wave t finishes row tile t: lane (j, g) has columns n0 + 4g .. + 3 of row 16 t + j
  const int r = wave * 16 + j, n = n0 + 4 * g;
  if (r >= a.R || n >= a.N) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < NW; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += s_acc[k][wave][lane][i];
  typedef Pack<T, 4> P4;
  typedef Pack<float, 4> F4;
  if (a.bias) {
    const P4 p = load_pack<T, 4>(reinterpret_cast<const T *>(a.bias) + n);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += E::to_float(p.v[i]);
  }
  P4 o;
  if constexpr (OUT == kStore) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = E::from_float(activate(v[i], a.act));
    store_pack<T, 4>(reinterpret_cast<T *>(a.y) + r * a.y_stride + n, o);
  } else if constexpr (OUT == kResidualF32) {
    const P4 p = load_pack<T, 4>(reinterpret_cast<const T *>(a.res) + r * a.res_stride + n);
    F4 f;
#pragma unroll
    for (int i = 0; i < 4; ++i) f.v[i] = v[i] + E::to_float(p.v[i]);
    store_pack<float, 4>(reinterpret_cast<float *>(a.y) + r * a.y_stride + n, f);
  } else if constexpr (OUT == kAddF32) {
    const F4 p = load_pack<float, 4>(reinterpret_cast<const float *>(a.res) + r * a.res_stride + n);
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = E::from_float(v[i] + p.v[i]);
    store_pack<T, 4>(reinterpret_cast<T *>(a.y) + r * a.y_stride + n, o);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = E::from_float(v[i]);
    const int part = n / a.hidden, c = n - part * a.hidden;
    if (part == 2) {
      store_pack<T, 4>(reinterpret_cast<T *>(a.y) + r * a.y_stride + c, o);
      return;
    }
    const int h = c / a.D, d = c - h * a.D, pos = a.kv_lens[r];
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

template <int DT, int IN, int OUT, int NW>
static void launch_rows_linear(const RowsArgs &a, hipStream_t s) {
  const unsigned grid = (unsigned)ceil_div(a.N, 16);
  if (a.R <= 16) rows_linear_kernel<DT, IN, OUT, NW, 1><<<grid, NW * kWave, 0, s>>>(a);
  else rows_linear_kernel<DT, IN, OUT, NW, 2><<<grid, NW * kWave, 0, s>>>(a);
}

// Waves per workgroup: about three steps of 64 channels each for narrow rows, so that all of a wave's weights are in flight
// at once; sixteen waves where K is long enough to keep them busy.
template <int DT, int IN, int OUT>
static int rows_linear(const RowsArgs &a, hipStream_t s) {
  const int64_t steps = ceil_div(a.K, 64);
  if (steps <= 16) launch_rows_linear<DT, IN, OUT, 4>(a, s);
  else if (IN != kPlain || steps <= 32) launch_rows_linear<DT, IN, OUT, 8>(a, s);
  else if constexpr (IN == kPlain) launch_rows_linear<DT, IN, OUT, 16>(a, s);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
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

  // k, v, q of the new tokens; K and V straight into the caches
  RowsArgs a{};
  a.x = p.x; a.x_stride = p.x_stride; a.R = R; a.K = (int)hid; a.N = (int)(3 * hid);
  a.w = p.qkv_weight; a.bias = p.qkv_bias; a.gamma = p.norm1_weight; a.beta = p.norm1_bias; a.eps = p.norm1_eps;
  a.y = q; a.y_stride = hid;
  a.k_cache = p.k_cache; a.v_cache = p.v_cache; a.kv_lens = p.kv_lens; a.hidden = (int)hid; a.D = p.size_per_head; a.Sk = p.cache_len;
  a.c_sb = p.cache_strides[0]; a.c_sh = p.cache_strides[1]; a.c_ss = p.cache_strides[2];
  a.page_table = p.page_table; a.max_pages = p.max_pages_per_seq; a.num_pages = p.num_pages;
  a.lg_page = p.page_table ? log2_page(p.page_size) : 0;
  int rc = rows_linear<DT, kNorm16, kScatterKVQ>(a, s);
  if (rc) return rc;
  // attention over the caches, the new position included
  rc = decode_attn_ahead(q, p.k_cache, p.v_cache, ctx, p.kv_lens, p.page_table, R, p.head_num, p.cache_len, p.max_pages_per_seq,
                         p.page_size, p.num_pages, p.size_per_head, p.cache_strides, p.scale, p.dtype, attn_ws, attn_bytes, s);
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
  if (p->batch > kMaxRows || hid > kMaxWidth || p->size_per_head % 8 || p->size_per_head > 512 || p->mlp_width % 8 || p->mlp_width > INT32_MAX)
    return EN_ERR_UNSUPPORTED;
  if (p->activation < EN_ACT_NONE || p->activation > EN_ACT_GELU) return EN_ERR_UNSUPPORTED;
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
