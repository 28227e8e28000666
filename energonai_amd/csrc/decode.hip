// Single-query attention contractions for cached decode: one new token per
// sequence against a ragged K/V cache.  Both are matrix-vector products whose
// cost is the K (or V) bytes streamed from HBM, so they are written as
// streaming reductions with 128-bit loads, one workgroup per (batch, head):
// LPK lanes cover one cached row of D elements, 256/LPK rows are in flight per
// step, four steps are unrolled so each lane keeps 64 bytes outstanding.
#include "common.hip.h"

namespace en {

struct DecodeArgs {
  const void *x;    // q [B,H,D] (QK) or p [B,H,Smax] (PV)
  const void *kv;   // cache [B,H,Smax,D], strided
  void *out;        // scores [B,H,Smax] (QK) or ctx [B,H,D] (PV)
  const int32_t *kv_lens;
  int H, Sk, D;
  int64_t sb, sh, ss;
  float alpha;
  int stream;       // the cache is too large to stay in the memory-side cache: read it with non-temporal loads
};

// A cache that cannot stay in the 256 MB memory-side cache between steps is streamed with
// non-temporal loads (measured on a 2.4 GB cache: QK 5.1 -> 5.8 TB/s, PV 5.6 -> 6.3 TB/s).
constexpr int64_t kStreamCacheBytes = 256ll << 20;
// ... and by workgroups of 1024 lanes per (batch, head): more rows of one cache in flight per workgroup
// (same cache: QK 5.8 -> 6.2 TB/s, PV 6.3 -> 6.8 TB/s over 256 lanes; 64 lanes: 4.1 / 4.5 TB/s)
constexpr int kStreamBlock = 1024;

template <int DT, int LPK, bool STREAM>
__global__ __launch_bounds__(STREAM ? kStreamBlock : kBlock) void decode_qk_kernel(DecodeArgs a) {
  constexpr int kBlock = STREAM ? kStreamBlock : en::kBlock;
  typedef Elem<DT> E;
  typedef typename E::T T;
  constexpr int EPV = 16 / E::kSize;
  constexpr int KPS = kBlock / LPK;  // keys per step
  constexpr int U = 4;
  const int h = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x;
  const int c = tid % LPK, slot = tid / LPK;
  const int kl = min(a.kv_lens[b], a.Sk);
  const T *q = reinterpret_cast<const T *>(a.x) + ((int64_t)b * a.H + h) * a.D;
  const T *kbase = reinterpret_cast<const T *>(a.kv) + (int64_t)b * a.sb + (int64_t)h * a.sh;
  T *srow = reinterpret_cast<T *>(a.out) + ((int64_t)b * a.H + h) * a.Sk;

  // head sizes that are not a power-of-two number of vectors (80, 96) run on the next power of two of
  // lanes per key; the lanes past the head load nothing and add zeros
  const bool cv = c * EPV < a.D;
  float qv[EPV];
  {
    Pack<T, EPV> pk;
#pragma unroll
    for (int e = 0; e < EPV; ++e) pk.v[e] = E::from_float(0.f);
    if (cv) pk = load_pack<T, EPV>(q + c * EPV);
#pragma unroll
    for (int e = 0; e < EPV; ++e) qv[e] = E::to_float(pk.v[e]) * a.alpha;
  }
  for (int k0 = 0; k0 < kl; k0 += KPS * U) {  // uniform trip count: all lanes reach the reductions
    Pack<T, EPV> kv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = k0 + u * KPS + slot;
      if (key < kl && cv) kv[u] = __builtin_bit_cast(Pack<T, EPV>, load16<STREAM>(kbase + (int64_t)key * a.ss + c * EPV));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = k0 + u * KPS + slot;
      float dot = 0.f;
      if (key < kl && cv) {
#pragma unroll
        for (int e = 0; e < EPV; ++e) dot += qv[e] * E::to_float(kv[u].v[e]);
      }
      dot = group_allreduce<OpSum, LPK>(dot);
      if (c == 0 && key < kl) srow[key] = E::from_float(dot);
    }
  }
}

template <int DT, int LPK, bool STREAM>
__global__ __launch_bounds__(STREAM ? kStreamBlock : kBlock) void decode_pv_kernel(DecodeArgs a) {
  constexpr int kBlock = STREAM ? kStreamBlock : en::kBlock;
  typedef Elem<DT> E;
  typedef typename E::T T;
  constexpr int EPV = 16 / E::kSize;
  constexpr int KPS = kBlock / LPK;
  constexpr int U = 4;
  __shared__ float s_acc[KPS][LPK * EPV + 1];
  const int h = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x;
  const int c = tid % LPK, slot = tid / LPK;
  const int kl = min(a.kv_lens[b], a.Sk);
  const T *prow = reinterpret_cast<const T *>(a.x) + ((int64_t)b * a.H + h) * a.Sk;
  const T *vbase = reinterpret_cast<const T *>(a.kv) + (int64_t)b * a.sb + (int64_t)h * a.sh;
  T *ctx = reinterpret_cast<T *>(a.out) + ((int64_t)b * a.H + h) * a.D;
  const bool cv = c * EPV < a.D;     // lanes past the head size idle (head sizes such as 80 and 96)

  float acc[EPV];
#pragma unroll
  for (int e = 0; e < EPV; ++e) acc[e] = 0.f;
  for (int k0 = slot; k0 < kl; k0 += KPS * U) {
    Pack<T, EPV> vv[U];
    float p[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = k0 + u * KPS;
      p[u] = 0.f;
      if (key < kl && cv) {
        vv[u] = __builtin_bit_cast(Pack<T, EPV>, load16<STREAM>(vbase + (int64_t)key * a.ss + c * EPV));
        p[u] = E::to_float(prow[key]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = k0 + u * KPS;
      if (key < kl && cv) {
#pragma unroll
        for (int e = 0; e < EPV; ++e) acc[e] += p[u] * E::to_float(vv[u].v[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < EPV; ++e) s_acc[slot][c * EPV + e] = acc[e];
  __syncthreads();
  for (int d = tid; d < a.D; d += kBlock) {
    float s = 0.f;
#pragma unroll 4
    for (int j = 0; j < KPS; ++j) s += s_acc[j][d];
    ctx[d] = E::from_float(s);
  }
}

template <int DT, template <int, int> class Launcher>
static int dispatch_lpk(const DecodeArgs &a, int batch, hipStream_t s) {
  constexpr int EPV = 16 / Elem<DT>::kSize;
  int lpk = 4;                                 // lanes per key: vectors in a head, rounded up to a power of two
  while (lpk * EPV < a.D) lpk *= 2;
  dim3 grid((unsigned)a.H, (unsigned)batch, 1);
  switch (lpk) {
    case 4: Launcher<DT, 4>::go(a, grid, s); break;
    case 8: Launcher<DT, 8>::go(a, grid, s); break;
    case 16: Launcher<DT, 16>::go(a, grid, s); break;
    case 32: Launcher<DT, 32>::go(a, grid, s); break;
    case 64: Launcher<DT, 64>::go(a, grid, s); break;
    default: return EN_ERR_UNSUPPORTED;
  }
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

template <int DT, int LPK> struct QkLauncher {
  static void go(const DecodeArgs &a, dim3 grid, hipStream_t s) {
    if (a.stream) decode_qk_kernel<DT, LPK, true><<<grid, kStreamBlock, 0, s>>>(a);
    else decode_qk_kernel<DT, LPK, false><<<grid, kBlock, 0, s>>>(a);
  }
};
template <int DT, int LPK> struct PvLauncher {
  static void go(const DecodeArgs &a, dim3 grid, hipStream_t s) {
    if (a.stream) decode_pv_kernel<DT, LPK, true><<<grid, kStreamBlock, 0, s>>>(a);
    else decode_pv_kernel<DT, LPK, false><<<grid, kBlock, 0, s>>>(a);
  }
};

static int64_t cache_bytes(int batch, int head_num, int k_seq_len, int size_per_head, int dtype) {
  return (int64_t)batch * head_num * k_seq_len * size_per_head * dtype_size(dtype);
}

static int check_decode(const void *x, const void *kv, const void *out, const int32_t *lens, int batch, int head_num,
                        int k_seq_len, int size_per_head, int64_t sb, int64_t sh, int64_t ss, int dtype) {
  if (!x || !kv || !out || !lens) return EN_ERR_NULL;
  if (batch < 1 || batch > 65535 || head_num < 1 || k_seq_len < 1 || size_per_head < 1) return EN_ERR_SHAPE;
  const int es = dtype_size(dtype);
  if (!es) return EN_ERR_DTYPE;
  const int epv = 16 / es;
  if ((size_per_head % epv) != 0) return EN_ERR_UNSUPPORTED;
  if (!aligned_to(kv, 16) || (sb % epv) || (sh % epv) || (ss % epv)) return EN_ERR_ALIGN;
  return EN_OK;
}

}  // namespace en

namespace en {

// ---------------------------------------------------------------------------------------------------------------
// Single-pass decode attention: ctx = softmax(scale * q K^T) V for one query per sequence, K and V each read
// once, scores and probabilities never written.  One workgroup per (batch, head); LPK lanes cover one cached row
// (16 bytes each), so the workgroup's NT / LPK lane groups take U * NT / LPK keys per stage.  Two stages of registers:
// the K and V pieces of the next one are in flight while this one's are worked on.  Bound by the reads of the caches
// (large batches: 6.8 TB/s, what a kernel that only reads reaches) and, for small batches, by what a launch costs before
// its first byte arrives and after its last (an empty launch 2.8 us, 16 keys 4.4 us).  NT and U: see AttnForm.
// Each lane group carries its own running maximum, sum and output slice (online softmax, maximum and exponent in the
// log2 domain with the scale folded in).  At the end the groups of a wave are combined in registers and the waves
// through LDS: every group through LDS (33 KB, one lane per channel adding up 64 rows) took 2 us of a workgroup's life
// and left no room for a third workgroup (72 units of 1655 keys, unsplit: 38 -> 21.8 us at 1024 x 1).
// The sequences are taken longest first (rank computed inside each workgroup from the lengths, batches of up to
// kRankBatch): the launch then ends on its short units instead of on whatever the last batch index happens to hold.
// ---------------------------------------------------------------------------------------------------------------
struct DecodeAttnArgs {
  const void *q;      // [B,H,D]
  const void *k, *v;  // caches [B,H,Smax,D], strided
  void *ctx;          // [B,H,D]
  const int32_t *kv_lens;
  int B, H, Sk, D;
  int64_t k_sb, k_sh, k_ss, v_sb, v_sh, v_ss;
  float c_exp;        // scale * log2(e)
  int nsplit;         // workgroups that share one (batch, head) unit's keys (grid z); 1: none
  // nsplit > 1, share z of unit u at u * nsplit + z: its unnormalised output [B*H*nsplit][D], and behind all of those its
  // maximum (log2 domain) and sum [B*H*nsplit][2]
  float *partial;
  // paged caches: k and v are pools of pages, page p of head h at p * k_sb + h * k_sh (k_sb is the page stride),
  // position s of sequence b in page page_table[b * max_pages + s / page] at row s % page
  const int32_t *page_table;
  int max_pages, lg_page, num_pages;
  int len_add;        // 1: the newest token sits at position kv_lens[b] already, the length does not count it yet
  int ranked;         // sequences are taken longest first
};

__device__ __forceinline__ int cached_len(const DecodeAttnArgs &a, int b) { return max(min(a.kv_lens[b] + a.len_add, a.Sk), 0); }

// Keys of one workgroup when nsplit share a unit: a multiple of 64, so that the keys of one wave (at most 16) never
// straddle a share or a page.  The combine kernel derives the same shares from the length.
__device__ __forceinline__ int split_share(int kl, int nsplit) {
  return nsplit > 1 ? ((kl + nsplit - 1) / nsplit + 63) & ~63 : kl;
}

constexpr int kRankBatch = 256;

// N floats of a workspace, which is 4-byte aligned and no more; the hardware takes wide accesses at such addresses.
template <int N> struct Partial {
  typedef float type __attribute__((ext_vector_type(N), aligned(4)));
};
template <> struct Partial<1> {
  typedef float type;
};

__device__ __forceinline__ Partial<2>::type *partial_ml(const DecodeAttnArgs &a, int64_t share_index) {
  return reinterpret_cast<Partial<2>::type *>(a.partial + (int64_t)a.B * a.H * a.nsplit * a.D) + share_index;
}

// From this size on (K and V together) the single pass reads the caches with non-temporal loads: a step walks the caches
// of every layer before it comes back to these, and four layers of 64 MB are the whole memory-side cache (61 MB read
// cold: 14.1 -> 13.2 us; 18 MB still in that cache: 6.3 -> 6.7 us; 192 MB of 768 units x 64, walked full 29.4 -> 26.2 us, with
// 1..40 keys in each sequence, which stay in the cache whatever its capacity, 6.1 -> 6.5 us).
constexpr int64_t kAttnStreamBytes = 64ll << 20;

// Sum or maximum over the lane groups of a wave (lanes that hold the same channels): every lane ends with the result.
// Rows of 16 lanes are swapped with permlane swaps, groups of 8 and 4 lanes inside a row rotated with DPP: no LDS.
template <typename Op, int LPK>
__device__ __forceinline__ float across_groups(float v) {
  if (LPK <= 4) v = Op::apply(v, dpp_move<0x124>(v));   // row_ror:4
  if (LPK <= 8) v = Op::apply(v, dpp_move<0x128>(v));   // row_ror:8
  if (LPK <= 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = Op::apply(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  if (LPK <= 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = Op::apply(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return v;
}

// The residual + LayerNorm of a decode step behind the attention, in its launch, where few units leave the launch short and a
// second one, its start and the trip through the caches are much of what the step consists of.  Nobody waits: the workgroups of a
// sequence count themselves at a word once their results are where every XCD sees them, and the last one normalises the
// sequence's row, combining the shares of each unit first where keys are shared.  It leaves the word at zero.
struct DecodeTail {
  const void *residual, *gamma, *beta;
  void *y;
  uint32_t *words;      // one a sequence, kTailWordStride apart
  int hidden;
  float eps;
};
constexpr int kTailWordStride = 16;       // a 64-byte line each
constexpr int kTailVectors = 2;           // 16-byte vectors of a row a lane takes
constexpr int kAgentScope = 16;           // cache policy of an access that all XCDs see (sc1)

template <typename T>
__device__ __forceinline__ void store_agent(T *p, T v) {
  if constexpr (sizeof(T) == 2)
    __hip_atomic_store(reinterpret_cast<uint16_t *>(p), __builtin_bit_cast(uint16_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else
    __hip_atomic_store(reinterpret_cast<uint32_t *>(p), __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_agent(const float *p) {
  return __uint_as_float(__hip_atomic_load(reinterpret_cast<const uint32_t *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Called by the whole workgroup behind its agent-scope stores: true in the last of `all` workgroups.
__device__ __forceinline__ bool last_to_arrive(uint32_t *word, int all, int *s_last) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the wave's results are where every XCD sees them ...
  lds_barrier();                                        // ... and the other waves' too, before the workgroup counts itself
  if (threadIdx.x == 0) {
    const bool last = (int)atomicAdd(word, 1u) == all - 1;
    if (last) __hip_atomic_store(word, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *s_last = last;
  }
  lds_barrier();
  return *s_last != 0;
}

template <int N, bool AGENT = false>
__device__ __forceinline__ void combine_shares(const DecodeAttnArgs &a, int b, int64_t unit, int d, float (&out)[N]);

// y = LayerNorm(x + residual) of sequence b's row; x is the context, or (SHARED) what its units' shares combine to, four channels a
// lane.
template <int DT, int NT, bool SHARED>
__device__ __forceinline__ void tail_row(const DecodeAttnArgs &a, const DecodeTail &n, int b, float *s_a, float *s_b) {
  typedef Elem<DT> E;
  typedef typename E::T T;
  constexpr int N = SHARED ? 4 : 16 / E::kSize, VPL = SHARED ? 1 : kTailVectors;
  typedef Pack<T, N> P;
  const int tid = threadIdx.x, nvec = n.hidden / N;
  const int64_t row = (int64_t)b * n.hidden;
  const rsrc_t ctx = make_rsrc(reinterpret_cast<const T *>(a.ctx) + row, (uint32_t)(n.hidden * E::kSize));
  uint4 raw[VPL];
  P r[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = min(tid + NT * j, nvec - 1) * N;
    if constexpr (!SHARED) raw[j] = buffer_load16<kAgentScope>(ctx, (uint32_t)(v * E::kSize));
    r[j] = load_pack<T, N>(reinterpret_cast<const T *>(n.residual) + row + v);
  }
  float x[VPL][N], s = 0.f, d2 = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const bool in = tid + NT * j < nvec;
    if constexpr (SHARED) {
      const int v = min(tid, nvec - 1) * N, h = v / a.D;
      combine_shares<N, true>(a, b, (int64_t)b * a.H + h, v - h * a.D, x[j]);
    } else {
      const P c = __builtin_bit_cast(P, raw[j]);
#pragma unroll
      for (int e = 0; e < N; ++e) x[j][e] = E::to_float(c.v[e]);
    }
#pragma unroll
    for (int e = 0; e < N; ++e) {
      x[j][e] = in ? x[j][e] + E::to_float(r[j].v[e]) : 0.f;
      s += x[j][e];
    }
  }
  const float mu = block_allreduce<OpSum, NT / kWave>(s, s_a) / (float)n.hidden;
#pragma unroll
  for (int j = 0; j < VPL; ++j)
    if (tid + NT * j < nvec)
#pragma unroll
      for (int e = 0; e < N; ++e) d2 += (x[j][e] - mu) * (x[j][e] - mu);
  const float inv = 1.0f / sqrtf(block_allreduce<OpSum, NT / kWave>(d2, s_b) / (float)n.hidden + n.eps);
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = (tid + NT * j) * N;
    if (tid + NT * j < nvec) {
      const P g = load_pack<T, N>(reinterpret_cast<const T *>(n.gamma) + v), bt = load_pack<T, N>(reinterpret_cast<const T *>(n.beta) + v);
      P o;
#pragma unroll
      for (int e = 0; e < N; ++e) o.v[e] = E::from_float((x[j][e] - mu) * inv * E::to_float(g.v[e]) + E::to_float(bt.v[e]));
      store_pack<T, N>(reinterpret_cast<T *>(n.y) + row + v, o);
    }
  }
}

template <int DT, int LPK, int NT, int U, bool STREAM, bool PAGED, bool TAIL>
__device__ __forceinline__ void decode_attn_unit(const DecodeAttnArgs &a, const DecodeTail *tail) {
  typedef Elem<DT> E;
  typedef typename E::T T;
  constexpr int EPV = 16 / E::kSize;
  constexpr int G = NT / LPK;        // lane groups = keys per step
  constexpr int NW = NT / kWave;
  constexpr int W = LPK * EPV;       // channels the lanes of a group cover (>= D)
  __shared__ float s_m[NW], s_l[NW];
  __shared__ float s_acc[NW][W];
  __shared__ int s_len[kRankBatch];
  __shared__ int s_b;
  const int tid = threadIdx.x;
  const int h = blockIdx.x;
  int b = blockIdx.y;
  if (a.ranked) {
    // batch index whose length ranks blockIdx.y-th (longest first, ties by index)
    for (int i = tid; i < a.B; i += NT) s_len[i] = cached_len(a, i);
    __syncthreads();
    for (int i = tid; i < a.B; i += NT) {
      const int mine = s_len[i];
      int rank = 0;
      for (int j = 0; j < a.B; ++j) {
        const int lj = s_len[j];
        rank += (lj > mine || (lj == mine && j < i)) ? 1 : 0;
      }
      if (rank == (int)blockIdx.y) s_b = i;
    }
    __syncthreads();
    b = __builtin_amdgcn_readfirstlane(s_b);      // lengths, bounds and the walk through the pages stay scalar
  }
  const int c = tid % LPK, g = tid / LPK;
  const int kl = cached_len(a, b);
  // with the keys of a unit split over nsplit workgroups this one takes [kbeg, kend); a share past the end has no
  // workgroup's worth of work and leaves no partial (the combine kernel derives the same shares from the length)
  const int share = split_share(kl, a.nsplit);
  const int kbeg = (int)blockIdx.z * share, kend = min(kl, kbeg + share);
  if (a.nsplit > 1 && kbeg >= kl && !(TAIL && blockIdx.z == 0)) return;      // an empty sequence has a row to normalise as well
  const T *q = reinterpret_cast<const T *>(a.q) + ((int64_t)b * a.H + h) * a.D;
  const T *kbase = reinterpret_cast<const T *>(a.k) + (PAGED ? 0 : (int64_t)b * a.k_sb) + (int64_t)h * a.k_sh;
  const T *vbase = reinterpret_cast<const T *>(a.v) + (PAGED ? 0 : (int64_t)b * a.v_sb) + (int64_t)h * a.v_sh;
  T *ctx = reinterpret_cast<T *>(a.ctx) + ((int64_t)b * a.H + h) * a.D;
  const bool cv = c * EPV < a.D;     // lanes past the head size idle (head sizes such as 80 and 96)

  float qv[EPV];
  {
    Pack<T, EPV> pk;
#pragma unroll
    for (int e = 0; e < EPV; ++e) pk.v[e] = E::from_float(0.f);
    if (cv) pk = load_pack<T, EPV>(q + c * EPV);
#pragma unroll
    for (int e = 0; e < EPV; ++e) qv[e] = E::to_float(pk.v[e]) * a.c_exp;
  }
  float m_run = -INFINITY, l_run = 0.f;
  float acc[EPV];
#pragma unroll
  for (int e = 0; e < EPV; ++e) acc[e] = 0.f;

  // Bounds-checked buffer loads: a row at or past the sequence's length (and a lane past the head size) reads
  // zeros without a branch, so the loads of the next stage can be issued ahead of this stage's arithmetic and the
  // compiler counts what is outstanding statically.
  const rsrc_t k_rsrc = make_rsrc(kbase, kl > 0 ? (uint32_t)(((int64_t)(kl - 1) * a.k_ss + a.D) * E::kSize) : 0u);
  const rsrc_t v_rsrc = make_rsrc(vbase, kl > 0 ? (uint32_t)(((int64_t)(kl - 1) * a.v_ss + a.D) * E::kSize) : 0u);
  const uint32_t k_row = (uint32_t)(a.k_ss * E::kSize), v_row = (uint32_t)(a.v_ss * E::kSize);
  const uint32_t col = cv ? (uint32_t)(c * 16) : kOutOfRange;
  constexpr int AUX = STREAM ? 2 : 0;
  // Paged caches: the keys of one wave (64 / LPK of them, first one a multiple of that) lie in one page, so the
  // page is a wave-uniform choice of buffer.  Each wave keeps the ids of 64 pages of the sequence in one register,
  // lane i the id of page tab0 + i, and takes the one it needs with a lane read; the register is filled again when
  // the walk leaves its range (every 64 pages).  An id outside the pool makes an empty buffer: zeros, no access.
  constexpr int KPW = kWave / LPK;                   // keys of one wave and step
  const int wkey = __builtin_amdgcn_readfirstlane(tid / kWave) * KPW;
  const uint32_t page_mask = PAGED ? (1u << a.lg_page) - 1u : 0u;
  const uint32_t k_page_bytes = PAGED ? (uint32_t)((((int64_t)page_mask) * a.k_ss + a.D) * E::kSize) : 0u;
  const uint32_t v_page_bytes = PAGED ? (uint32_t)((((int64_t)page_mask) * a.v_ss + a.D) * E::kSize) : 0u;
  int tab = -1, tab0 = 0;
  auto fill_tab = [&](int first_page) {
    tab0 = first_page;
    const int pi = first_page + (tid % kWave);
    tab = pi < a.max_pages ? a.page_table[(int64_t)b * a.max_pages + pi] : -1;
    // waited for here: left outstanding into the loop, every key's page lookup would wait for all K and V loads before it
    // (72 heads x 128, pages of 64: 576 units of 2048 keys 120.4 -> 105.2 us, of 8192 464.6 -> 404.3, 72 of 2048 26.9 -> 19.2)
    asm volatile("" : "+v"(tab));
  };
  if constexpr (PAGED) fill_tab((kbeg + wkey) >> a.lg_page);
  auto load_stage = [&](uint4 (&kk)[U], uint4 (&vv)[U], int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = k0 + u * G + g;
      const uint32_t in = key < kend ? 0u : kOutOfRange;     // past the end: out of range whatever the stride
      if constexpr (PAGED) {
        const int pi = (k0 + u * G + wkey) >> a.lg_page;      // wave-uniform
        if (pi - tab0 >= kWave) fill_tab(pi);
        const int id = __builtin_amdgcn_readlane(tab, pi - tab0);
        const bool ok = (unsigned)id < (unsigned)a.num_pages;
        const rsrc_t kr = make_rsrc(kbase + (int64_t)id * a.k_sb, ok ? k_page_bytes : 0u);
        const rsrc_t vr = make_rsrc(vbase + (int64_t)id * a.v_sb, ok ? v_page_bytes : 0u);
        const uint32_t row = (uint32_t)key & page_mask;
        kk[u] = buffer_load16<AUX>(kr, row * k_row + col | in);
        vv[u] = buffer_load16<AUX>(vr, row * v_row + col | in);
      } else {
        kk[u] = buffer_load16<AUX>(k_rsrc, (uint32_t)key * k_row + col | in);
        vv[u] = buffer_load16<AUX>(v_rsrc, (uint32_t)key * v_row + col | in);
      }
    }
  };
  auto compute_stage = [&](const uint4 (&kk)[U], const uint4 (&vv)[U], int k0) {
    float sc[U];
    float m_new = m_run;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = k0 + u * G + g;
      const Pack<T, EPV> kp = __builtin_bit_cast(Pack<T, EPV>, kk[u]);
      float dot = 0.f;
#pragma unroll
      for (int e = 0; e < EPV; ++e) dot += qv[e] * E::to_float(kp.v[e]);
      dot = group_allreduce<OpSum, LPK>(dot);
      sc[u] = key < kend ? dot : -INFINITY;
      m_new = fmaxf(m_new, sc[u]);
    }
    if (m_new > -INFINITY) {            // this group has seen a key: (-inf) - (-inf) never reaches exp2
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);      // exp2(-inf) = 0 on the first key
      l_run *= alpha;
#pragma unroll
      for (int e = 0; e < EPV; ++e) acc[e] *= alpha;
      m_run = m_new;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const Pack<T, EPV> vp = __builtin_bit_cast(Pack<T, EPV>, vv[u]);
        const float p = __builtin_amdgcn_exp2f(sc[u] - m_new);        // 0 for a key past the end
        l_run += p;
#pragma unroll
        for (int e = 0; e < EPV; ++e) acc[e] += p * E::to_float(vp.v[e]);
      }
    }
  };
  // NS stages of registers: while one is worked on, the loads of the others are in flight
  constexpr int STEP = G * U;
  constexpr int NS = 2;
  static_assert((2 * NS - 1) * STEP <= 4096, "the host check allows 4096 keys past the end");
  uint4 kr[NS][U], vr[NS][U];
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) load_stage(kr[st], vr[st], kbeg + st * STEP);
  for (int k0 = kbeg; k0 < kend; k0 += NS * STEP) {   // uniform trip count: all lanes reach the reductions
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      load_stage(kr[(st + NS - 1) % NS], vr[(st + NS - 1) % NS], k0 + (st + NS - 1) * STEP);
      // one key per lane group and stage: a wave whose keys of this stage are all past the end has nothing to do
      if (U > 1 || k0 + st * STEP + wkey < kend) compute_stage(kr[st], vr[st], k0 + st * STEP);
    }
  }
  // the lane groups of a wave share one maximum, add up in registers, and the waves combine through LDS
  const float m_w = across_groups<OpMax, LPK>(m_run);
  const float scale_g = m_run > -INFINITY ? __builtin_amdgcn_exp2f(m_run - m_w) : 0.f;
  l_run = across_groups<OpSum, LPK>(l_run * scale_g);
#pragma unroll
  for (int e = 0; e < EPV; ++e) acc[e] = across_groups<OpSum, LPK>(acc[e] * scale_g);
  const int lane = tid % kWave, wave = tid / kWave;
  if (lane < LPK) {
#pragma unroll
    for (int e = 0; e < EPV; ++e) s_acc[wave][c * EPV + e] = acc[e];
    if (lane == 0) { s_m[wave] = m_w; s_l[wave] = l_run; }
  }
  __syncthreads();
  const int64_t share_index = ((int64_t)b * a.H + h) * a.nsplit + blockIdx.z;
  for (int d = tid; d < a.D; d += NT) {
    float m_all = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) m_all = fmaxf(m_all, s_m[w]);
    float l = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = s_m[w] > -INFINITY ? __builtin_amdgcn_exp2f(s_m[w] - m_all) : 0.f;
      l += s_l[w] * f;
      o += s_acc[w][d] * f;
    }
    if (a.nsplit > 1) {
      if constexpr (TAIL) {
        store_agent(a.partial + share_index * a.D + d, o);
        if (d == 0) {
          float *ml = reinterpret_cast<float *>(partial_ml(a, share_index));
          store_agent(ml, m_all);
          store_agent(ml + 1, l);
        }
      } else {
        a.partial[share_index * a.D + d] = o;
        if (d == 0) *partial_ml(a, share_index) = Partial<2>::type{m_all, l};
      }
    } else {
      const T c_d = E::from_float(l > 0.f ? o / l : 0.f);
      if constexpr (TAIL) store_agent(ctx + d, c_d);
      else ctx[d] = c_d;
    }
  }
  if constexpr (TAIL) {
    __shared__ int s_last;
    // workgroups of a sequence: a unit's shares that had keys, one for an empty sequence
    const int shares = a.nsplit > 1 && share > 0 ? (kl + share - 1) / share : 1;
    if (!last_to_arrive(tail->words + b * kTailWordStride, a.H * shares, &s_last)) return;
    if (a.nsplit > 1) tail_row<DT, NT, true>(a, *tail, b, s_m, s_l);
    else tail_row<DT, NT, false>(a, *tail, b, s_m, s_l);
  }
}

template <int DT, int LPK, int NT, int U, bool STREAM, bool PAGED = false>
__global__ __launch_bounds__(NT, U == 1 ? 8 : 4) void decode_attn_kernel(DecodeAttnArgs a) {
  decode_attn_unit<DT, LPK, NT, U, STREAM, PAGED, false>(a, nullptr);
}
// At most two units a CU: registers for four waves a SIMD are enough, and the row at the end needs them.
template <int DT, int LPK, int NT, int U, bool STREAM>
__global__ __launch_bounds__(NT, 4) void decode_attn_norm_kernel(DecodeAttnArgs a, DecodeTail tail) {
  decode_attn_unit<DT, LPK, NT, U, STREAM, false, true>(a, &tail);
}

// Combines N channels, from channel d on, of the partial results of a unit's shares.  The partials of kAhead shares are
// sent for together with the length that says how many of them were written (the workspace holds nsplit of them whatever
// the length), so that one trip to memory is waited for instead of three.
// AGENT: other workgroups of the same launch wrote them.
template <int N, bool AGENT>
__device__ __forceinline__ void combine_shares(const DecodeAttnArgs &a, int b, int64_t unit, int d, float (&out)[N]) {
  constexpr int kAhead = 4;
  typedef typename Partial<N>::type P;
  float m_run = -INFINITY, l_run = 0.f;
#pragma unroll
  for (int e = 0; e < N; ++e) out[e] = 0.f;
  int nvalid = a.nsplit;
  for (int z0 = 0; z0 < nvalid; z0 += kAhead) {
    Partial<2>::type ml[kAhead];
    P o[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int64_t share_index = unit * a.nsplit + min(z0 + i, a.nsplit - 1);
      if constexpr (AGENT) {
        static_assert(N == 4, "one 16-byte load");
        const float *p_ml = reinterpret_cast<const float *>(partial_ml(a, share_index));
        o[i] = __builtin_bit_cast(P, buffer_load16<kAgentScope>(make_rsrc(a.partial, 0x7fffffffu), (uint32_t)((share_index * a.D + d) * 4)));
        ml[i] = Partial<2>::type{load_agent(p_ml), load_agent(p_ml + 1)};
      } else {
        o[i] = *reinterpret_cast<const P *>(a.partial + share_index * a.D + d);
        ml[i] = *partial_ml(a, share_index);
      }
    }
    if (z0 == 0) {
      const int kl = cached_len(a, b);
      const int share = split_share(kl, a.nsplit);
      nvalid = share > 0 ? (kl + share - 1) / share : 0;       // shares that had keys
    }
    float m_new = m_run;
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (z0 + i >= nvalid) ml[i].x = -INFINITY;
      m_new = fmaxf(m_new, ml[i].x);
    }
    if (m_new == -INFINITY) continue;
    const float keep = __builtin_amdgcn_exp2f(m_run - m_new);        // exp2(-inf) = 0 before the first share
    l_run *= keep;
#pragma unroll
    for (int e = 0; e < N; ++e) out[e] *= keep;
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (ml[i].x == -INFINITY) continue;                            // never written, or no key: whatever it holds stays out
      const float f = __builtin_amdgcn_exp2f(ml[i].x - m_new);
      l_run += ml[i].y * f;
#pragma unroll
      for (int e = 0; e < N; ++e) {
        if constexpr (N == 1) out[e] += o[i] * f;
        else out[e] += o[i][e] * f;
      }
    }
    m_run = m_new;
  }
  const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
#pragma unroll
  for (int e = 0; e < N; ++e) out[e] *= inv;
}

template <int DT>
__global__ __launch_bounds__(kBlock) void decode_attn_combine_kernel(DecodeAttnArgs a) {
  typedef Elem<DT> E;
  typedef typename E::T T;
  const int unit = blockIdx.x, b = unit / a.H;
  T *ctx = reinterpret_cast<T *>(a.ctx) + (int64_t)unit * a.D;
  for (int d = threadIdx.x; d < a.D; d += kBlock) {
    float o[1];
    combine_shares<1>(a, b, unit, d, o);
    ctx[d] = E::from_float(o[0]);
  }
}

// The decode step whose shared units are followed by nothing but residual + LayerNorm (no projection in between, LayerNorm
// width = heads * size_per_head): the combine pass is the LayerNorm's input and has no launch or round trip of its own.
// One workgroup of 1024 lanes per sequence, four channels per lane and vector: a row of 9216 channels is 2.25 vectors.
// One sequence of 72 heads x 128, 1655 keys: combine + LayerNorm 4.8 + 3.5 us as two launches, one of 4.4.
struct DecodeNormArgs {
  DecodeAttnArgs attn;
  const void *residual, *gamma, *beta;
  void *y;
  int hidden;
  float eps;
};

constexpr int kNormLanes = 1024;

template <int DT, int VPL>
__global__ __launch_bounds__(kNormLanes) void decode_combine_norm_kernel(DecodeNormArgs n) {
  typedef Elem<DT> E;
  typedef typename E::T T;
  constexpr int N = 4;                 // channels per vector
  typedef Pack<T, N> P;
  __shared__ float s_a[kNormLanes / kWave], s_b[kNormLanes / kWave];
  const DecodeAttnArgs &a = n.attn;
  const int b = blockIdx.x, t = threadIdx.x;
  const int nvec = n.hidden / N;
  const T *res = reinterpret_cast<const T *>(n.residual) + (int64_t)b * n.hidden;
  const T *gamma = reinterpret_cast<const T *>(n.gamma), *beta = reinterpret_cast<const T *>(n.beta);
  P r[VPL], g[VPL], bt[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = min(t + kNormLanes * j, nvec - 1);
    r[j] = load_pack<T, N>(res + v * N);
    g[j] = load_pack<T, N>(gamma + v * N);
    bt[j] = load_pack<T, N>(beta + v * N);
  }
  float x[VPL][N];
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = t + kNormLanes * j;
    if (v < nvec) {
      const int h = v * N / a.D, d = v * N - h * a.D;
      combine_shares<N>(a, b, (int64_t)b * a.H + h, d, x[j]);
#pragma unroll
      for (int e = 0; e < N; ++e) {
        x[j][e] += E::to_float(r[j].v[e]);
        s += x[j][e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < N; ++e) x[j][e] = 0.f;
    }
  }
  s = block_allreduce<OpSum, kNormLanes / kWave>(s, s_a);
  const float mu = s / (float)n.hidden;
  float d2 = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j)
    if (t + kNormLanes * j < nvec)
#pragma unroll
      for (int e = 0; e < N; ++e) d2 += (x[j][e] - mu) * (x[j][e] - mu);
  d2 = block_allreduce<OpSum, kNormLanes / kWave>(d2, s_b);
  const float inv = 1.0f / sqrtf(d2 / (float)n.hidden + n.eps);
  T *y = reinterpret_cast<T *>(n.y) + (int64_t)b * n.hidden;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = t + kNormLanes * j;
    if (v < nvec) {
      P o;
#pragma unroll
      for (int e = 0; e < N; ++e)
        o.v[e] = E::from_float((x[j][e] - mu) * inv * E::to_float(g[j].v[e]) + E::to_float(bt[j].v[e]));
      store_pack<T, N>(y + v * N, o);
    }
  }
}

template <int DT>
static int launch_combine_norm(const DecodeNormArgs &n, hipStream_t s) {
  const int vpl = (int)ceil_div(n.hidden / 4, kNormLanes);
  const unsigned grid = (unsigned)n.attn.B;
  if (vpl <= 1) decode_combine_norm_kernel<DT, 1><<<grid, kNormLanes, 0, s>>>(n);
  else if (vpl == 2) decode_combine_norm_kernel<DT, 2><<<grid, kNormLanes, 0, s>>>(n);
  else if (vpl == 3) decode_combine_norm_kernel<DT, 3><<<grid, kNormLanes, 0, s>>>(n);
  else decode_combine_norm_kernel<DT, 4><<<grid, kNormLanes, 0, s>>>(n);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

// Which form of the kernel a call runs (lanes per workgroup x keys per lane group and stage; all hold two stages).  The host
// knows the capacity of the caches and not the lengths, so a form has to carry its range from caches that are nearly empty to
// full ones.  Kernel times per call, caches of several layers walked in turn; "1..40" are lengths of 1..40 keys.
//   kTiny   256 x 1   units that fill the chip on caches of few steps (a step: the keys 256 lanes take at once): what counts is
//                     that all workgroups are resident (64 registers, eight waves a SIMD) and that a wave without keys left
//                     does nothing.  1920 units x 64 fp16, capacity 128: 1..40 7.7 us, 32..128 12.9 (256 x 2: 10.0, 13.9;
//                     512 x 4: 22.1, 26.3); capacity 512: 7.7, 128..512 30.3 (10.5, 29.1; 23.3, 36.3).  Where
//                     few workgroups walk far, one key ahead is too few: 512 units x 64, 1..1024 keys 17.2 (256 x 2: 15.6), 768
//                     units x 128, 1..2048 keys 76.3 (512 x 4: 70.2).
//   kSmall  256 x 2   the keys of few units are shared between workgroups, or the caches are short: start-up and the
//                     final combination count.  72 units of 1655 keys (61 MB), four shares each, without the combine
//                     kernel: 13.2 us against 17.2 for 1024 x 1, 15.0 for 512 x 2; 96 units of ~70 keys 4.4 us.
//   kPair   512 x 2   keys are shared and there are fewer workgroups than CUs: 48 units x 128, two shares of 700 keys each, fp16
//                     13.7 us, fp32 19.4 with the combine kernel (256 x 2: 18.2, 27.8), 12 units x 64, 1024 keys, fp16 6.9 (7.1);
//                     nearly empty caches 0.4 us more.  Or the keys of 256..511 units in long shares, three and more workgroups
//                     a CU: 384 units x 128, 1..2048 keys, fp32 74.3 us, fp16 41.3 (82.7, 45.2), 1..4096 147, 82 (162, 88).
//   kDeep   512 x 4   enough units for the chip but not many rounds of them, long caches: more bytes in flight per workgroup.
//                     768 units of 1..4000 keys 113.9 us (512 x 2: 116.1, 256 x 4: 116.0).  Nearly empty caches pay for it:
//                     768 units x 128, capacity 2048, 1..40 fp16 13.5 us (256 x 4: 8.8, 1024 x 1: 12.2).
//   kMany   256 x 4   between those two, many units, and few units on caches too short to share: 768 units x 64, 1..2048
//                     keys 39.3 us (512 x 4: 40.6, 256 x 1: 41.1); 4608 units of 1..2048 keys (2.6 GB) 388 us, 6.8 TB/s
//                     (512 x 4: 396, 1024 x 1: 402); 72 units of 512 keys 7.9 us (256 x 2: 10.4).
// Up to one unit a CU none waits for another, whatever their order: the lengths of the whole batch, two barriers and the ranks
// are saved (8 sequences x 12 heads x 64 of 100 keys 5.0 -> 4.4 us).
constexpr int64_t kUnrankedUnits = 256;

enum class AttnForm { kTiny, kSmall, kPair, kDeep, kMany };

static AttnForm attn_form(const DecodeAttnArgs &a, int lpk) {
  const int64_t units = (int64_t)a.B * a.H;
  const int64_t steps = ceil_div(ceil_div(a.Sk, a.nsplit) * lpk, kBlock);      // of a workgroup, caches full
  if (a.nsplit > 1) return units * a.nsplit < 256 || (units >= 256 && steps > 32) ? AttnForm::kPair : AttnForm::kSmall;
  if (units < 256) return a.Sk <= 256 ? AttnForm::kSmall : AttnForm::kMany;
  if (units < 512) return steps <= 8 ? AttnForm::kTiny : a.Sk <= 256 || steps <= 16 ? AttnForm::kSmall : AttnForm::kMany;
  if (steps <= 32) return steps <= 16 || units >= 768 ? AttnForm::kTiny : AttnForm::kSmall;
  return units < 2048 && steps > 64 ? AttnForm::kDeep : AttnForm::kMany;
}

template <int DT, int LPK, bool PAGED, int NT, int U>
static void launch_attn(const DecodeAttnArgs &a, dim3 grid, bool stream_cache, hipStream_t s) {
  DecodeAttnArgs args = a;
  args.ranked = a.nsplit == 1 && a.B > 1 && a.B <= kRankBatch && (int64_t)a.B * a.H > kUnrankedUnits;
  if (stream_cache) decode_attn_kernel<DT, LPK, NT, U, true, PAGED><<<grid, NT, 0, s>>>(args);
  else decode_attn_kernel<DT, LPK, NT, U, false, PAGED><<<grid, NT, 0, s>>>(args);
}

template <int DT, int LPK, bool PAGED>
static void launch_attn_form(const DecodeAttnArgs &a, dim3 grid, bool stream_cache, hipStream_t s) {
  switch (attn_form(a, LPK)) {
    case AttnForm::kTiny: launch_attn<DT, LPK, PAGED, 256, 1>(a, grid, stream_cache, s); break;
    case AttnForm::kSmall: launch_attn<DT, LPK, PAGED, 256, 2>(a, grid, stream_cache, s); break;
    case AttnForm::kPair: launch_attn<DT, LPK, PAGED, 512, 2>(a, grid, stream_cache, s); break;
    case AttnForm::kDeep: launch_attn<DT, LPK, PAGED, 512, 4>(a, grid, stream_cache, s); break;
    default: launch_attn<DT, LPK, PAGED, 256, 4>(a, grid, stream_cache, s); break;
  }
}

template <int DT, bool PAGED = false>
static int dispatch_attn(const DecodeAttnArgs &a, bool stream_cache, hipStream_t s, bool combine = true) {
  constexpr int EPV = 16 / Elem<DT>::kSize;
  int lpk = 4;
  while (lpk * EPV < a.D) lpk *= 2;
  dim3 grid((unsigned)a.H, (unsigned)a.B, (unsigned)a.nsplit);
  switch (lpk) {
    case 4: launch_attn_form<DT, 4, PAGED>(a, grid, stream_cache, s); break;
    case 8: launch_attn_form<DT, 8, PAGED>(a, grid, stream_cache, s); break;
    case 16: launch_attn_form<DT, 16, PAGED>(a, grid, stream_cache, s); break;
    case 32: launch_attn_form<DT, 32, PAGED>(a, grid, stream_cache, s); break;
    case 64: launch_attn_form<DT, 64, PAGED>(a, grid, stream_cache, s); break;
    default: return EN_ERR_UNSUPPORTED;
  }
  EN_RETURN_IF_LAUNCH_FAILED();
  if (a.nsplit > 1 && combine) {
    decode_attn_combine_kernel<DT><<<(unsigned)(a.B * a.H), kBlock, 0, s>>>(a);
    EN_RETURN_IF_LAUNCH_FAILED();
  }
  return EN_OK;
}

template <int DT, int LPK, int NT, int U>
static void launch_attn_norm(const DecodeAttnArgs &a, const DecodeTail &tail, dim3 grid, bool stream_cache, hipStream_t s) {
  DecodeAttnArgs args = a;
  args.ranked = a.nsplit == 1 && a.B > 1 && a.B <= kRankBatch && (int64_t)a.B * a.H > kUnrankedUnits;
  if (stream_cache) decode_attn_norm_kernel<DT, LPK, NT, U, true><<<grid, NT, 0, s>>>(args, tail);
  else decode_attn_norm_kernel<DT, LPK, NT, U, false><<<grid, NT, 0, s>>>(args, tail);
}

// Whether a decode layer is one launch: the forms of attn_form below 512 units, for heads of 33..128 channels (fp32: 17..128).  From
// 512 units on the attention is several times what the second launch costs.
static bool one_launch_takes(const DecodeAttnArgs &a, int elem_size) {
  const int epv = 16 / elem_size;
  if (a.B > kRankBatch || (int64_t)a.B * a.H >= 512 || a.D % epv || a.D <= 4 * epv || a.D > 128) return false;
  int lpk = 8;
  while (lpk * epv < a.D) lpk *= 2;
  const int64_t hidden = (int64_t)a.H * a.D, lanes = attn_form(a, lpk) == AttnForm::kPair ? 512 : 256;
  // One workgroup has the whole row to read.  us a layer of a decode loop, two launches / one, where the host's second launch is most
  // of what is saved (in brackets the GPU alone): 1 x 12 heads x 64, up to 300 keys 8.5 / 6.1 (6.2 / 6.1), 8 x 12 x 64 8.5 / 6.4
  // (6.9 / 6.4), 2 x 8 x 64 fp32, up to 800 9.2 / 8.0, 16 x 24 x 64, up to 900 15.8 / 15.0 (15.8 / 15.0), 16 x 32 x 128, up to 128
  // 10.1 / 10.1; of five vectors a lane, 2 x 60 x 128, up to 500 10.3 / 10.7, 5 x 72 x 128 35.8 / 36.8.  Rows of shares are four
  // channels a lane, sixteen bytes from each share: 1 x 5 x 64, 4000 keys 9.3 / 7.5 (7.9 / 7.5), 10 x 16 x 64, up to 2000 15.5 / 14.3
  // (15.4 / 14.3); combined unit by unit in front of the row, which takes wider ones, 6 x 64 x 128 41.9 / 43.9.
  return a.nsplit > 1 ? hidden <= 4 * lanes : hidden * elem_size <= kTailVectors * 16 * lanes;
}

template <int DT, int LPK>
static int launch_attn_norm_form(const DecodeAttnArgs &a, const DecodeTail &tail, dim3 grid, bool stream_cache, hipStream_t s) {
  switch (attn_form(a, LPK)) {
    case AttnForm::kTiny: launch_attn_norm<DT, LPK, 256, 1>(a, tail, grid, stream_cache, s); break;
    case AttnForm::kSmall: launch_attn_norm<DT, LPK, 256, 2>(a, tail, grid, stream_cache, s); break;
    case AttnForm::kPair: launch_attn_norm<DT, LPK, 512, 2>(a, tail, grid, stream_cache, s); break;
    case AttnForm::kMany: launch_attn_norm<DT, LPK, 256, 4>(a, tail, grid, stream_cache, s); break;
    default: return EN_ERR_UNSUPPORTED;
  }
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

template <int DT>
static int dispatch_attn_norm(const DecodeAttnArgs &a, const DecodeTail &tail, bool stream_cache, hipStream_t s) {
  constexpr int EPV = 16 / Elem<DT>::kSize;
  const dim3 grid((unsigned)a.H, (unsigned)a.B, (unsigned)a.nsplit);
  if constexpr (DT == EN_F32)
    if (a.D > 16 * EPV) return launch_attn_norm_form<DT, 32>(a, tail, grid, stream_cache, s);
  if (a.D > 8 * EPV) return launch_attn_norm_form<DT, 16>(a, tail, grid, stream_cache, s);
  return launch_attn_norm_form<DT, 8>(a, tail, grid, stream_cache, s);
}

// How many workgroups share one unit's keys: none while the units alone fill the chip (512 units and more); else
// enough for about four workgroups per CU, each share at least 512 keys long (shorter shares cost more in start-up
// and in the combine pass than they win: 22 us instead of 25 for one sequence of 2048 keys).
static int decode_split(int batch, int head_num, int k_seq_len) {
  constexpr int kTargetWorkgroups = 1024, kMinShare = 512;
  const int64_t units = (int64_t)batch * head_num;
  if (units >= 512 || k_seq_len < 2 * kMinShare) return 1;
  int64_t n = (kTargetWorkgroups + units - 1) / units;
  if (n > k_seq_len / kMinShare) n = k_seq_len / kMinShare;
  if (n > 64) n = 64;
  return n < 1 ? 1 : (int)n;
}

// Appends one new K row and one new V row per (batch, head) to the caches at position
// kv_lens[b]; sequences whose cache is full are left alone and counted.  Bytes are moved as they are.
struct AppendArgs {
  const unsigned char *k_new, *v_new;
  unsigned char *k_cache, *v_cache;
  const int32_t *kv_lens;
  int H, Sk;
  int row_bytes;
  int64_t n_sb, n_sh;           // strides of the new rows, bytes
  int64_t c_sb, c_sh, c_ss;     // strides of the caches, bytes
  int32_t *overflow;            // counts the sequences that had no room (null: not counted)
};

template <typename Vec>
__global__ __launch_bounds__(kWave) void kv_append_kernel(AppendArgs a) {
  const int h = blockIdx.x, b = blockIdx.y;
  const int pos = a.kv_lens[b];
  if (pos < 0 || pos >= a.Sk) {
    if (a.overflow && h == 0 && threadIdx.x == 0) atomicAdd(a.overflow, 1);
    return;
  }
  const int64_t src = (int64_t)b * a.n_sb + (int64_t)h * a.n_sh;
  const int64_t dst = (int64_t)b * a.c_sb + (int64_t)h * a.c_sh + (int64_t)pos * a.c_ss;
  for (int i = threadIdx.x * (int)sizeof(Vec); i < a.row_bytes; i += kWave * (int)sizeof(Vec)) {
    *reinterpret_cast<Vec *>(a.k_cache + dst + i) = *reinterpret_cast<const Vec *>(a.k_new + src + i);
    *reinterpret_cast<Vec *>(a.v_cache + dst + i) = *reinterpret_cast<const Vec *>(a.v_new + src + i);
  }
}


// Paged caches: the same append, the row found through the page table.  A sequence whose next position has no page
// (position past max_pages * page, id outside the pool) is left alone and counted.
struct PagedAppendArgs {
  const unsigned char *k_new, *v_new;
  unsigned char *k_pool, *v_pool;
  const int32_t *kv_lens, *page_table;
  int H, max_pages, lg_page, num_pages;
  int row_bytes;
  int64_t n_sb, n_sh;           // strides of the new rows, bytes
  int64_t p_sp, p_sh, p_ss;     // page, head and row strides of the pools, bytes
  int32_t *overflow;
};

__global__ __launch_bounds__(kWave) void kv_append_paged_kernel(PagedAppendArgs a) {
  const int h = blockIdx.x, b = blockIdx.y;
  const int pos = a.kv_lens[b];
  const int pi = pos >> a.lg_page;
  const int id = (pos >= 0 && pi < a.max_pages) ? a.page_table[(int64_t)b * a.max_pages + pi] : -1;
  if ((unsigned)id >= (unsigned)a.num_pages) {
    if (a.overflow && h == 0 && threadIdx.x == 0) atomicAdd(a.overflow, 1);
    return;
  }
  const int64_t src = (int64_t)b * a.n_sb + (int64_t)h * a.n_sh;
  const int64_t dst = (int64_t)id * a.p_sp + (int64_t)h * a.p_sh + (int64_t)(pos & ((1 << a.lg_page) - 1)) * a.p_ss;
  for (int i = threadIdx.x * 16; i < a.row_bytes; i += kWave * 16) {
    *reinterpret_cast<uint4 *>(a.k_pool + dst + i) = *reinterpret_cast<const uint4 *>(a.k_new + src + i);
    *reinterpret_cast<uint4 *>(a.v_pool + dst + i) = *reinterpret_cast<const uint4 *>(a.v_new + src + i);
  }
}

// Prefill into pages: the rows of sequence b, packed tokens cu[b] .. of a [T, src_head_rows, D] source of which heads
// src_head_first .. + H - 1 are taken, go to rows 0 .. len - 1 of the sequence's pages.
struct PagedFillArgs {
  const unsigned char *src;
  unsigned char *pool;
  const int32_t *cu, *page_table;
  int H, S, max_pages, lg_page, num_pages;
  int vecs_per_row;             // 16-byte vectors per head row
  int64_t s_row, s_head;        // source: bytes per token, bytes per head row
  int64_t head_first_bytes;
  int64_t p_sp, p_sh, p_ss;
  int32_t *overflow;
};

__global__ __launch_bounds__(kBlock) void kv_fill_paged_kernel(PagedFillArgs a) {
  constexpr int ROWS = 4;
  const int b = blockIdx.y;
  const int t0 = a.cu[b], len = min(a.cu[b + 1] - t0, a.S);
  const int per_row = a.H * a.vecs_per_row;
  for (int r = 0; r < ROWS; ++r) {
    const int s = blockIdx.x * ROWS + r;
    if (s >= len) return;
    const int pi = s >> a.lg_page;
    const int id = pi < a.max_pages ? a.page_table[(int64_t)b * a.max_pages + pi] : -1;
    if ((unsigned)id >= (unsigned)a.num_pages) {
      if (a.overflow && threadIdx.x == 0) atomicAdd(a.overflow, 1);
      continue;
    }
    const unsigned char *src = a.src + (int64_t)(t0 + s) * a.s_row + a.head_first_bytes;
    unsigned char *dst = a.pool + (int64_t)id * a.p_sp + (int64_t)(s & ((1 << a.lg_page) - 1)) * a.p_ss;
    for (int i = threadIdx.x; i < per_row; i += kBlock) {
      const int h = i / a.vecs_per_row, c = i - h * a.vecs_per_row;
      *reinterpret_cast<uint4 *>(dst + (int64_t)h * a.p_sh + c * 16) =
          *reinterpret_cast<const uint4 *>(src + (int64_t)h * a.s_head + c * 16);
    }
  }
}

static int log2_exact(int v) {
  int lg = 0;
  while ((1 << lg) < v) ++lg;
  return (1 << lg) == v ? lg : -1;
}

// Checks the arguments of the contiguous-cache entry points and fills the kernel's.
static int attn_args(DecodeAttnArgs &a, const void *q, const void *k_cache, const void *v_cache, void *ctx,
                     const int32_t *kv_lens, int batch, int head_num, int k_seq_len, int size_per_head,
                     const int64_t *k_strides, const int64_t *v_strides, float scale, int dtype, void *workspace,
                     int64_t workspace_bytes) {
  if (!k_strides || !v_strides || !v_cache) return EN_ERR_NULL;
  int rc = check_decode(q, k_cache, ctx, kv_lens, batch, head_num, k_seq_len, size_per_head, k_strides[0], k_strides[1],
                        k_strides[2], dtype);
  if (rc) return rc;
  const int es = dtype_size(dtype), epv = 16 / es;
  if (!aligned_to(v_cache, 16) || (v_strides[0] % epv) || (v_strides[1] % epv) || (v_strides[2] % epv)) return EN_ERR_ALIGN;
  if (!aligned_to(q, 16) || !aligned_to(ctx, es)) return EN_ERR_ALIGN;
  if (size_per_head > 64 * epv) return EN_ERR_UNSUPPORTED;
  // 32-bit byte offsets inside a (batch, head) unit, two stages of keys past the end included
  if (((int64_t)k_seq_len + 4096) * k_strides[2] * es >= (1ll << 31) || ((int64_t)k_seq_len + 4096) * v_strides[2] * es >= (1ll << 31))
    return EN_ERR_UNSUPPORTED;
  if (!(scale > 0.f)) return EN_ERR_UNSUPPORTED;     // the running maximum is kept in units of scale * log2(e)
  for (int i = 0; i < 3; ++i)
    if (k_strides[i] < 0 || v_strides[i] < 0) return EN_ERR_UNSUPPORTED;
  // a unit's keys are shared between workgroups only when the caller brought the room for their partial results
  const int64_t need = en_decode_attn_workspace_bytes(batch, head_num, k_seq_len, size_per_head);
  const bool split = need > 0 && workspace && workspace_bytes >= need && aligned_to(workspace, 4);
  a = DecodeAttnArgs{q, k_cache, v_cache, ctx, kv_lens, batch, head_num, k_seq_len, size_per_head, k_strides[0], k_strides[1],
                     k_strides[2], v_strides[0], v_strides[1], v_strides[2], scale * 1.4426950408889634f,
                     split ? decode_split(batch, head_num, k_seq_len) : 1, static_cast<float *>(workspace)};
  return EN_OK;
}

static int dispatch_attn_dtype(const DecodeAttnArgs &a, int dtype, hipStream_t s, bool combine) {
  const bool stream_cache = 2 * cache_bytes(a.B, a.H, a.Sk, a.D, dtype) >= kAttnStreamBytes;
  switch (dtype) {
    case EN_F32: return dispatch_attn<EN_F32>(a, stream_cache, s, combine);
    case EN_F16: return dispatch_attn<EN_F16>(a, stream_cache, s, combine);
    default: return dispatch_attn<EN_BF16>(a, stream_cache, s, combine);
  }
}

static int paged_attn_args(DecodeAttnArgs &a, const void *q, const void *k_pool, const void *v_pool, void *ctx,
                           const int32_t *kv_lens, const int32_t *page_table, int batch, int head_num, int max_pages_per_seq,
                           int page_size, int num_pages, int size_per_head, const int64_t *k_strides, const int64_t *v_strides,
                           float scale, int dtype, void *workspace, int64_t workspace_bytes) {
  if (!k_strides || !v_strides || !v_pool || !page_table) return EN_ERR_NULL;
  if (max_pages_per_seq < 1 || num_pages < 1) return EN_ERR_SHAPE;
  const int lg = log2_exact(page_size);
  if (lg < 4) return EN_ERR_UNSUPPORTED;                                  // a power of two, at least 16: a wave's keys share a page
  if ((int64_t)max_pages_per_seq * page_size >= (1ll << 30)) return EN_ERR_SHAPE;
  const int k_seq_len = max_pages_per_seq * page_size;
  int rc = check_decode(q, k_pool, ctx, kv_lens, batch, head_num, k_seq_len, size_per_head, k_strides[0], k_strides[1],
                        k_strides[2], dtype);
  if (rc) return rc;
  const int es = dtype_size(dtype), epv = 16 / es;
  if (!aligned_to(v_pool, 16) || (v_strides[0] % epv) || (v_strides[1] % epv) || (v_strides[2] % epv)) return EN_ERR_ALIGN;
  if (!aligned_to(q, 16) || !aligned_to(ctx, es)) return EN_ERR_ALIGN;
  if (size_per_head > 64 * epv) return EN_ERR_UNSUPPORTED;
  // 32-bit byte offsets inside a page
  if ((int64_t)page_size * k_strides[2] * es >= (1ll << 31) || (int64_t)page_size * v_strides[2] * es >= (1ll << 31))
    return EN_ERR_UNSUPPORTED;
  if (!(scale > 0.f)) return EN_ERR_UNSUPPORTED;
  for (int i = 0; i < 3; ++i)
    if (k_strides[i] < 0 || v_strides[i] < 0) return EN_ERR_UNSUPPORTED;
  const int64_t need = en_decode_attn_workspace_bytes(batch, head_num, k_seq_len, size_per_head);
  const bool split = need > 0 && workspace && workspace_bytes >= need && aligned_to(workspace, 4);
  a = DecodeAttnArgs{q, k_pool, v_pool, ctx, kv_lens, batch, head_num, k_seq_len, size_per_head, k_strides[0], k_strides[1],
                     k_strides[2], v_strides[0], v_strides[1], v_strides[2], scale * 1.4426950408889634f,
                     split ? decode_split(batch, head_num, k_seq_len) : 1, static_cast<float *>(workspace),
                     page_table, max_pages_per_seq, lg, num_pages};
  return EN_OK;
}

static int dispatch_paged_dtype(const DecodeAttnArgs &a, int dtype, hipStream_t s) {
  const bool stream_cache = 2 * cache_bytes(a.B, a.H, a.Sk, a.D, dtype) >= kAttnStreamBytes;
  switch (dtype) {
    case EN_F32: return dispatch_attn<EN_F32, true>(a, stream_cache, s);
    case EN_F16: return dispatch_attn<EN_F16, true>(a, stream_cache, s);
    default: return dispatch_attn<EN_BF16, true>(a, stream_cache, s);
  }
}

int decode_attn_ahead(const void *q, const void *k_cache, const void *v_cache, void *ctx, const int32_t *kv_lens,
                      const int32_t *page_table, int batch, int head_num, int cache_len, int max_pages_per_seq, int page_size,
                      int num_pages, int size_per_head, const int64_t *strides, float scale, int dtype, void *workspace,
                      int64_t workspace_bytes, bool launch, hipStream_t stream) {
  DecodeAttnArgs a;
  const int rc = page_table ? paged_attn_args(a, q, k_cache, v_cache, ctx, kv_lens, page_table, batch, head_num, max_pages_per_seq,
                                              page_size, num_pages, size_per_head, strides, strides, scale, dtype, workspace,
                                              workspace_bytes)
                            : attn_args(a, q, k_cache, v_cache, ctx, kv_lens, batch, head_num, cache_len, size_per_head, strides,
                                        strides, scale, dtype, workspace, workspace_bytes);
  if (rc || !launch) return rc;
  a.len_add = 1;
  return page_table ? dispatch_paged_dtype(a, dtype, stream) : dispatch_attn_dtype(a, dtype, stream, true);
}

}  // namespace en

extern "C" {

int en_kv_append(const void *k_new, const void *v_new, void *k_cache, void *v_cache, const int32_t *kv_lens,
                 int batch, int head_num, int k_seq_len, int size_per_head, int64_t new_stride_b,
                 int64_t new_stride_h, int64_t cache_stride_b, int64_t cache_stride_h, int64_t cache_stride_s,
                 int elem_size, int32_t *overflow, en_stream_t stream) {
  using namespace en;
  if (!k_new || !v_new || !k_cache || !v_cache || !kv_lens) return EN_ERR_NULL;
  if (overflow && !aligned_to(overflow, 4)) return EN_ERR_ALIGN;
  if (elem_size != 2 && elem_size != 4) return EN_ERR_DTYPE;
  if (batch < 1 || head_num < 1 || k_seq_len < 1 || size_per_head < 1) return EN_ERR_SHAPE;
  if (batch > 65535) return EN_ERR_SHAPE;
  if (new_stride_b < 0 || new_stride_h < 0 || cache_stride_b < 0 || cache_stride_h < 0 || cache_stride_s < 0)
    return EN_ERR_UNSUPPORTED;
  AppendArgs a{(const unsigned char *)k_new, (const unsigned char *)v_new, (unsigned char *)k_cache,
               (unsigned char *)v_cache, kv_lens, head_num, k_seq_len, size_per_head * elem_size,
               new_stride_b * elem_size, new_stride_h * elem_size, cache_stride_b * elem_size,
               cache_stride_h * elem_size, cache_stride_s * elem_size, overflow};
  const dim3 grid((unsigned)head_num, (unsigned)batch, 1);
  hipStream_t s = (hipStream_t)stream;
  const bool v16 = (a.row_bytes % 16 == 0) && aligned_to(k_new, 16) && aligned_to(v_new, 16) &&
                   aligned_to(k_cache, 16) && aligned_to(v_cache, 16) && a.n_sb % 16 == 0 && a.n_sh % 16 == 0 &&
                   a.c_sb % 16 == 0 && a.c_sh % 16 == 0 && a.c_ss % 16 == 0;
  if (v16) {
    kv_append_kernel<uint4><<<grid, kWave, 0, s>>>(a);
  } else if (elem_size == 4) {
    if (!aligned_to(k_new, 4) || !aligned_to(v_new, 4) || !aligned_to(k_cache, 4) || !aligned_to(v_cache, 4))
      return EN_ERR_ALIGN;
    kv_append_kernel<uint32_t><<<grid, kWave, 0, s>>>(a);
  } else {
    if (!aligned_to(k_new, 2) || !aligned_to(v_new, 2) || !aligned_to(k_cache, 2) || !aligned_to(v_cache, 2))
      return EN_ERR_ALIGN;
    kv_append_kernel<uint16_t><<<grid, kWave, 0, s>>>(a);
  }
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

int64_t en_decode_attn_workspace_bytes(int batch, int head_num, int k_seq_len, int size_per_head) {
  using namespace en;
  if (batch < 1 || head_num < 1 || k_seq_len < 1 || size_per_head < 1) return 0;
  const int n = decode_split(batch, head_num, k_seq_len);
  return n > 1 ? (int64_t)batch * head_num * n * (size_per_head + 2) * (int64_t)sizeof(float) : 0;
}

int en_decode_attn(const void *q, const void *k_cache, const void *v_cache, void *ctx, const int32_t *kv_lens, int batch,
                   int head_num, int k_seq_len, int size_per_head, const int64_t *k_strides, const int64_t *v_strides,
                   float scale, int dtype, void *workspace, int64_t workspace_bytes, en_stream_t stream) {
  using namespace en;
  DecodeAttnArgs a;
  const int rc = attn_args(a, q, k_cache, v_cache, ctx, kv_lens, batch, head_num, k_seq_len, size_per_head, k_strides,
                           v_strides, scale, dtype, workspace, workspace_bytes);
  return rc ? rc : dispatch_attn_dtype(a, dtype, (hipStream_t)stream, true);
}

int en_decode_layer(const void *q, const void *k_cache, const void *v_cache, void *ctx, const int32_t *kv_lens, int batch,
                    int head_num, int k_seq_len, int size_per_head, const int64_t *k_strides, const int64_t *v_strides,
                    float scale, const void *dense_out, const void *residual, const void *gamma, const void *beta, void *y,
                    int64_t hidden, float eps, int dtype, int out_dtype, void *workspace, int64_t workspace_bytes,
                    en_stream_t stream) {
  using namespace en;
  if (!residual || !gamma || !beta || !y) return EN_ERR_NULL;
  if (hidden < 1 || (!dense_out && hidden != (int64_t)head_num * size_per_head)) return EN_ERR_SHAPE;
  DecodeAttnArgs a;
  int rc = attn_args(a, q, k_cache, v_cache, ctx, kv_lens, batch, head_num, k_seq_len, size_per_head, k_strides, v_strides,
                     scale, dtype, workspace, workspace_bytes);
  if (rc) return rc;
  const int vec = 4 * dtype_size(dtype);
  const bool one_pass = a.nsplit > 1 && !dense_out && out_dtype == dtype && hidden <= 4 * 4 * kNormLanes &&
                        aligned_to(residual, vec) && aligned_to(gamma, vec) && aligned_to(beta, vec) && aligned_to(y, vec);
  hipStream_t s = (hipStream_t)stream;
  rc = dispatch_attn_dtype(a, dtype, s, !one_pass);
  if (rc) return rc;
  if (!one_pass)
    return en_layernorm_fwd(y, nullptr, nullptr, nullptr, dense_out ? dense_out : ctx, residual, nullptr, gamma, beta, batch,
                            hidden, eps, dtype, out_dtype, stream);
  const DecodeNormArgs n{a, residual, gamma, beta, y, (int)hidden, eps};
  switch (dtype) {
    case EN_F32: return launch_combine_norm<EN_F32>(n, s);
    case EN_F16: return launch_combine_norm<EN_F16>(n, s);
    default: return launch_combine_norm<EN_BF16>(n, s);
  }
}

int en_decode_layer_norm_pays(int batch, int head_num, int k_seq_len, int size_per_head, int dtype) {
  using namespace en;
  const int es = dtype_size(dtype);
  if (!es || batch < 1 || head_num < 1 || k_seq_len < 1 || size_per_head < 1) return 0;
  DecodeAttnArgs a{};
  a.B = batch, a.H = head_num, a.Sk = k_seq_len, a.D = size_per_head, a.nsplit = decode_split(batch, head_num, k_seq_len);
  return one_launch_takes(a, es);
}

int64_t en_decode_layer_norm_words(void) { return (int64_t)en::kRankBatch * en::kTailWordStride; }

int en_decode_layer_norm(const void *q, const void *k_cache, const void *v_cache, void *ctx, const int32_t *kv_lens, int batch,
                         int head_num, int k_seq_len, int size_per_head, const int64_t *k_strides, const int64_t *v_strides,
                         float scale, const void *residual, const void *gamma, const void *beta, void *y, float eps, int dtype,
                         void *workspace, int64_t workspace_bytes, uint32_t *words, en_stream_t stream) {
  using namespace en;
  if (!residual || !gamma || !beta || !y || !words) return EN_ERR_NULL;
  DecodeAttnArgs a;
  const int rc = attn_args(a, q, k_cache, v_cache, ctx, kv_lens, batch, head_num, k_seq_len, size_per_head, k_strides, v_strides,
                           scale, dtype, workspace, workspace_bytes);
  if (rc) return rc;
  const int64_t es = dtype_size(dtype), hidden = (int64_t)head_num * size_per_head, rows = batch * hidden * es, S = k_seq_len;
  if (!one_launch_takes(a, (int)es)) return EN_ERR_UNSUPPORTED;
  for (const void *p : {(const void *)ctx, residual, gamma, beta, (const void *)y})
    if (!aligned_to(p, 16)) return EN_ERR_UNSUPPORTED;
  if (!aligned_to(words, 4) || (a.nsplit > 1 && !aligned_to(workspace, 16))) return EN_ERR_UNSUPPORTED;
  // A row is normalised while others are still attended to: buffers that a caller has laid over each other need two launches.
  auto cache = [&](const int64_t *st) { return ((batch - 1) * st[0] + (head_num - 1) * st[1] + (S - 1) * st[2] + size_per_head) * es; };
  struct Range { const void *p; int64_t bytes; };
  const Range read[] = {{q, rows}, {k_cache, cache(k_strides)}, {v_cache, cache(v_strides)}, {kv_lens, (int64_t)batch * 4},
                        {residual, rows}, {gamma, hidden * es}, {beta, hidden * es}};
  const Range written[] = {{y, rows}, {ctx, rows}, {workspace, a.nsplit > 1 ? workspace_bytes : 0}};
  auto meet = [](const Range &x, const Range &w) {
    const uintptr_t u = (uintptr_t)x.p, v = (uintptr_t)w.p;
    return u < v + (uintptr_t)w.bytes && v < u + (uintptr_t)x.bytes;
  };
  for (const Range &w : written)
    for (const Range &x : read)
      if (meet(x, w)) return EN_ERR_UNSUPPORTED;
  if (meet(written[0], written[1]) || meet(written[0], written[2]) || meet(written[1], written[2])) return EN_ERR_UNSUPPORTED;
  // A captured launch may run again on any stream, beside launches that use the same words.
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &capture) != hipSuccess) {      // e.g. the null stream beside a capture
    (void)hipGetLastError();
    return EN_ERR_UNSUPPORTED;
  }
  if (capture != hipStreamCaptureStatusNone) return EN_ERR_UNSUPPORTED;
  const DecodeTail tail{residual, gamma, beta, y, words, (int)hidden, eps};
  const bool stream_cache = 2 * cache_bytes(a.B, a.H, a.Sk, a.D, dtype) >= kAttnStreamBytes;
  switch (dtype) {
    case EN_F32: return dispatch_attn_norm<EN_F32>(a, tail, stream_cache, (hipStream_t)stream);
    case EN_F16: return dispatch_attn_norm<EN_F16>(a, tail, stream_cache, (hipStream_t)stream);
    default: return dispatch_attn_norm<EN_BF16>(a, tail, stream_cache, (hipStream_t)stream);
  }
}

int en_kv_append_paged(const void *k_new, const void *v_new, void *k_pool, void *v_pool, const int32_t *kv_lens,
                       const int32_t *page_table, int batch, int head_num, int max_pages_per_seq, int page_size,
                       int num_pages, int size_per_head, int64_t new_stride_b, int64_t new_stride_h,
                       const int64_t *pool_strides, int elem_size, int32_t *overflow, en_stream_t stream) {
  using namespace en;
  if (!k_new || !v_new || !k_pool || !v_pool || !kv_lens || !page_table || !pool_strides) return EN_ERR_NULL;
  if (overflow && !aligned_to(overflow, 4)) return EN_ERR_ALIGN;
  if (elem_size != 2 && elem_size != 4) return EN_ERR_DTYPE;
  if (batch < 1 || batch > 65535 || head_num < 1 || max_pages_per_seq < 1 || num_pages < 1 || size_per_head < 1) return EN_ERR_SHAPE;
  const int lg = log2_exact(page_size);
  if (lg < 4) return EN_ERR_UNSUPPORTED;                                  // a power of two, at least 16
  if ((int64_t)max_pages_per_seq * page_size >= (1ll << 31)) return EN_ERR_SHAPE;
  if (new_stride_b < 0 || new_stride_h < 0 || pool_strides[0] < 0 || pool_strides[1] < 0 || pool_strides[2] < 0)
    return EN_ERR_UNSUPPORTED;
  PagedAppendArgs a{(const unsigned char *)k_new, (const unsigned char *)v_new, (unsigned char *)k_pool,
                    (unsigned char *)v_pool, kv_lens, page_table, head_num, max_pages_per_seq, lg, num_pages,
                    size_per_head * elem_size, new_stride_b * elem_size, new_stride_h * elem_size,
                    pool_strides[0] * elem_size, pool_strides[1] * elem_size, pool_strides[2] * elem_size, overflow};
  if ((a.row_bytes % 16) || !aligned_to(k_new, 16) || !aligned_to(v_new, 16) || !aligned_to(k_pool, 16) ||
      !aligned_to(v_pool, 16) || (a.n_sb % 16) || (a.n_sh % 16) || (a.p_sp % 16) || (a.p_sh % 16) || (a.p_ss % 16))
    return EN_ERR_ALIGN;
  kv_append_paged_kernel<<<dim3((unsigned)head_num, (unsigned)batch, 1), kWave, 0, (hipStream_t)stream>>>(a);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

int en_kv_fill_paged(const void *src, void *pool, const int32_t *cu_seqlens, const int32_t *page_table, int batch,
                     int max_seq_len, int head_num, int size_per_head, int src_head_rows, int src_head_first,
                     int max_pages_per_seq, int page_size, int num_pages, const int64_t *pool_strides, int elem_size,
                     int32_t *overflow, en_stream_t stream) {
  using namespace en;
  if (!src || !pool || !cu_seqlens || !page_table || !pool_strides) return EN_ERR_NULL;
  if (overflow && !aligned_to(overflow, 4)) return EN_ERR_ALIGN;
  if (elem_size != 2 && elem_size != 4) return EN_ERR_DTYPE;
  if (batch < 1 || batch > 65535 || max_seq_len < 1 || head_num < 1 || size_per_head < 1 || max_pages_per_seq < 1 ||
      num_pages < 1)
    return EN_ERR_SHAPE;
  if (src_head_first < 0 || src_head_rows < src_head_first + head_num) return EN_ERR_SHAPE;
  const int lg = log2_exact(page_size);
  if (lg < 4) return EN_ERR_UNSUPPORTED;
  if ((int64_t)max_pages_per_seq * page_size >= (1ll << 31)) return EN_ERR_SHAPE;
  if (pool_strides[0] < 0 || pool_strides[1] < 0 || pool_strides[2] < 0) return EN_ERR_UNSUPPORTED;
  const int64_t row_bytes = (int64_t)size_per_head * elem_size;
  PagedFillArgs a{(const unsigned char *)src, (unsigned char *)pool, cu_seqlens, page_table, head_num, max_seq_len,
                  max_pages_per_seq, lg, num_pages, (int)(row_bytes / 16), (int64_t)src_head_rows * row_bytes, row_bytes,
                  (int64_t)src_head_first * row_bytes, pool_strides[0] * elem_size, pool_strides[1] * elem_size,
                  pool_strides[2] * elem_size, overflow};
  if ((row_bytes % 16) || !aligned_to(src, 16) || !aligned_to(pool, 16) || (a.p_sp % 16) || (a.p_sh % 16) || (a.p_ss % 16))
    return EN_ERR_ALIGN;
  const dim3 grid((unsigned)ceil_div(max_seq_len, 4), (unsigned)batch, 1);
  kv_fill_paged_kernel<<<grid, kBlock, 0, (hipStream_t)stream>>>(a);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

int en_decode_attn_paged(const void *q, const void *k_pool, const void *v_pool, void *ctx, const int32_t *kv_lens,
                         const int32_t *page_table, int batch, int head_num, int max_pages_per_seq, int page_size,
                         int num_pages, int size_per_head, const int64_t *k_strides, const int64_t *v_strides, float scale,
                         int dtype, void *workspace, int64_t workspace_bytes, en_stream_t stream) {
  using namespace en;
  DecodeAttnArgs a;
  const int rc = paged_attn_args(a, q, k_pool, v_pool, ctx, kv_lens, page_table, batch, head_num, max_pages_per_seq, page_size,
                                 num_pages, size_per_head, k_strides, v_strides, scale, dtype, workspace, workspace_bytes);
  return rc ? rc : dispatch_paged_dtype(a, dtype, (hipStream_t)stream);
}

int en_decode_qk(const void *q, const void *k_cache, void *scores, const int32_t *kv_lens, int batch, int head_num,
                 int k_seq_len, int size_per_head, int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_s,
                 float alpha, int dtype, en_stream_t stream) {
  using namespace en;
  int rc = check_decode(q, k_cache, scores, kv_lens, batch, head_num, k_seq_len, size_per_head, k_stride_b,
                        k_stride_h, k_stride_s, dtype);
  if (rc) return rc;
  if (!aligned_to(q, 16) || !aligned_to(scores, dtype_size(dtype))) return EN_ERR_ALIGN;
  DecodeArgs a{q, k_cache, scores, kv_lens, head_num, k_seq_len, size_per_head, k_stride_b, k_stride_h, k_stride_s,
               alpha, cache_bytes(batch, head_num, k_seq_len, size_per_head, dtype) >= kStreamCacheBytes};
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case EN_F32: return dispatch_lpk<EN_F32, QkLauncher>(a, batch, s);
    case EN_F16: return dispatch_lpk<EN_F16, QkLauncher>(a, batch, s);
    default: return dispatch_lpk<EN_BF16, QkLauncher>(a, batch, s);
  }
}

int en_decode_pv(const void *p, const void *v_cache, void *ctx, const int32_t *kv_lens, int batch, int head_num,
                 int k_seq_len, int size_per_head, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_s,
                 int dtype, en_stream_t stream) {
  using namespace en;
  int rc = check_decode(p, v_cache, ctx, kv_lens, batch, head_num, k_seq_len, size_per_head, v_stride_b, v_stride_h,
                        v_stride_s, dtype);
  if (rc) return rc;
  if (!aligned_to(p, dtype_size(dtype)) || !aligned_to(ctx, dtype_size(dtype))) return EN_ERR_ALIGN;
  DecodeArgs a{p, v_cache, ctx, kv_lens, head_num, k_seq_len, size_per_head, v_stride_b, v_stride_h, v_stride_s, 1.f,
               cache_bytes(batch, head_num, k_seq_len, size_per_head, dtype) >= kStreamCacheBytes};
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case EN_F32: return dispatch_lpk<EN_F32, PvLauncher>(a, batch, s);
    case EN_F16: return dispatch_lpk<EN_F16, PvLauncher>(a, batch, s);
    default: return dispatch_lpk<EN_BF16, PvLauncher>(a, batch, s);
  }
}

}  // extern "C"
