// Fused attention for fp32 storage (heads of up to 64 channels, the BERT-base shape of the reference's CPU
// path, examples/bert/bert.py:108-119 in fp32; wider ones have the second kernel below): ctx = softmax(scale * Q K^T, mask) V in one kernel, no score
// tensor.  The 16-bit kernels of fused.hip are built around 16-bit operand vectors (probabilities as 16-bit B
// operands, the transposing LDS read); here everything is fp32 on the 32x32x2 MFMA.
//
// Workgroup: 4 waves, one tile of 64 query rows of one (batch, head).  Wave (wq, wk): query rows 32 wq .. + 31 and
// the keys 32 wk .. + 31 of every 64-key tile, so the two waves of a query half split the keys between them, each
// with its own running maximum, sum and output (online softmax over its own keys only: no exchange per tile);
// the pair is combined once, through LDS, at the end.  Small problems are what this kernel is for (fp32 batches are
// short), and they are bound by the length of a workgroup's dependent chain: half the keys per wave halve it, and
// 64-row tiles give twice the workgroups of the 128-row tiles of the 16-bit kernels.
//
//   S^T = K Q^T      A = the wave's 32 K rows from LDS, B = Q fragments in registers; one query per lane.
//   online softmax   as in fused.hip (in-lane reductions, one exchange between the wave's halves, lazy rescale).
//   O^T += V^T P^T   B = the probabilities as they sit in the S^T accumulators (fp32, no conversion): the MFMA step
//                    for register (j, i) contracts over the two keys 8j + i and 8j + 4 + i that the lane's two
//                    halves hold; A = V at those keys, one channel per lane, read from the row-major V tile.
#include "fused_common.hip.h"

#include <type_traits>

namespace en {

// A wave's 32 keys of the online softmax: the scores of this lane's query (register 4j + i: key 8j + i of the lane's half) become
// probabilities over the running maximum; returns the sum of the lane's own.  `seen`: keys from the half's first on that the query
// sees; `all`: the wave's queries see every key.  The maximum moves only where a tile's lies above it by more than 8 in the exponent of two,
// and from -inf with the first tile: the gap stays finite where the scale is so small that 8 over it is not.
template <int DMT>
__device__ __forceinline__ float softmax_f32_keys(floatx16 &s, floatx16 (&o)[DMT], float &m_run, float &l_run, int seen, bool all, float c_exp) {
  const float lazy_gap = fminf(8.0f / c_exp, 1e30f);
  float m_tile = -INFINITY;
  if (all) {
#pragma unroll
    for (int x = 0; x < 16; ++x) m_tile = fmaxf(m_tile, s[x]);
  } else {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const float v = (8 * (x >> 2) + (x & 3) < seen) ? s[x] : -INFINITY;
      s[x] = v;
      m_tile = fmaxf(m_tile, v);
    }
  }
  float lo, hi;
  halves_of(m_tile, lo, hi);
  m_tile = fmaxf(lo, hi);
  if (__builtin_amdgcn_ballot_w64(m_tile - lazy_gap > m_run) != 0) {
    const float m_new = fmaxf(m_run, m_tile);
    const float alpha = (m_run == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((m_run - m_new) * c_exp);
    l_run *= alpha;
#pragma unroll
    for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
      for (int x = 0; x < 16; ++x) o[mt][x] *= alpha;
    m_run = m_new;
  }
  const float moff = (m_run == -INFINITY) ? 0.f : -m_run * c_exp;
  float l_tile = 0.f;
#pragma unroll
  for (int x = 0; x < 16; ++x) {
    s[x] = __builtin_amdgcn_exp2f(fmaf(s[x], c_exp, moff));       // exp2(-inf) = 0: masked keys
    l_tile += s[x];
  }
  return l_tile;
}

// What two waves that saw disjoint keys are weighed with: the factors of this wave's and the other's output, the sum of both and its inverse.
struct PairWeights {
  float mine, other, sum, inv;
};
__device__ __forceinline__ PairWeights pair_weights(float m0, float l0, float m1, float l1, float c_exp) {
  const float m = fmaxf(m0, m1);
  const float w0 = (m0 == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((m0 - m) * c_exp);
  const float w1 = (m1 == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((m1 - m) * c_exp);
  const float l = l0 * w0 + l1 * w1;
  return {w0, w1, l, l > 0.f ? 1.0f / l : 0.f};
}

template <int DP, bool NORM>
__device__ __forceinline__ void fused_f32_tile(const FusedArgs &fa, const NormArgs *norm) {
  typedef float T;
  typedef Mma<EN_F32> M;
  const AttnArgs &a = fa.base;
  constexpr int EPV = 4;
  constexpr int BK = 64;                         // keys per tile (32 per wave)
  constexpr int NVS = DP / M::KPV;               // 128-bit steps over the head dim
  constexpr int DMT = DP / 32;                   // 32-channel MFMA tiles of the output
  constexpr int KP = DP + 4;                     // LDS pitch of a K row: 16-byte fragment reads of 32 rows spread over the banks
  constexpr int VP = DP + 8;                     // LDS pitch of a V row: the wave's halves read rows four keys apart, 4 VP = 32 (mod 64) banks
  constexpr int VEC_ROW = DP / EPV;
  constexpr int LOADS = BK * VEC_ROW / kBlock;   // 128-bit loads per lane and tile, for each of K and V
  constexpr float kLog2e = 1.4426950408889634f;
  static_assert(DP == 64, "pitches and the combine area are laid out for 64 channels");
  __shared__ __attribute__((aligned(16))) float lds_k[BK * KP];
  __shared__ __attribute__((aligned(16))) float lds_v[BK * VP];

  const int unit = blockIdx.y, qi = blockIdx.x;
  const int b = unit / a.H, h = unit % a.H;
  const SeqAhead ahead = seq_ahead(a, fa.q_row0, fa.k_row0);
  const Seq seq = seq_of(a, ahead, b, fa.q_row0, fa.k_row0);
  const int kl = seq.kl, ql = seq.ql;
  const int q0 = qi * kF32QTile;
  if (q0 >= ql) return;
  const int nk = tile_key_extent(a, min(q0 + kF32QTile, ql) - 1, kl, ql);
  const int nkt = (nk + BK - 1) / BK;
  NormTile rows;
  if constexpr (NORM) rows = norm_tile_of(*norm, (int64_t)b * gridDim.x + qi, seq.q_row + q0, min(kF32QTile, ql - q0), h, a.H);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, g = lane >> 5;
  const int wq = wave & 1, wk = wave >> 1;
  const int q_first = q0 + wq * 32;
  const int q_lane = q_first + r;
  // keys this lane's query may see, and the wave's smallest and largest such extent
  const int vis_l = (q_lane < ql) ? (a.causal ? min(kl, q_lane + (kl - ql) + 1) : kl) : 0;
  const int vis_min = (q_first + 31 < ql) ? (a.causal ? min(kl, q_first + (kl - ql) + 1) : kl) : 0;
  const int vis_max = (q_first < ql) ? (a.causal ? min(kl, min(q_first + 31, ql - 1) + (kl - ql) + 1) : kl) : 0;

  const int64_t qr = seq.q_row, kr = seq.k_row;
  const T *qbase = reinterpret_cast<const T *>(a.a_ptr) + (int64_t)b * a.q_sb + qr * a.q_ss + (int64_t)h * a.q_sh;
  const T *kbase = reinterpret_cast<const T *>(a.b_ptr) + (int64_t)b * a.k_sb + kr * a.k_ss + (int64_t)h * a.k_sh;
  const T *vbase = reinterpret_cast<const T *>(fa.v) + (int64_t)b * fa.v_sb + kr * fa.v_ss + (int64_t)h * fa.v_sh;
  T *cbase = reinterpret_cast<T *>(a.out) + (int64_t)b * fa.c_sb + qr * fa.c_ss + (int64_t)h * fa.c_sh;

  // Q fragments: this lane's query row, four channels per step (rows past the last valid one are never stored)
  uint4 qf[NVS];
  {
    const T *qrow = qbase + (int64_t)min(q_lane, ql - 1) * a.q_ss;
#pragma unroll
    for (int vs = 0; vs < NVS; ++vs) {
      const int d = M::k_of(vs, g, NVS);
      qf[vs] = (d < a.D) ? *reinterpret_cast<const uint4 *>(qrow + d) : zero4();
    }
  }

  // K / V tiles come through registers (bounds-checked: rows at or past the last key and channels past the head
  // size read as zeros) a tile ahead of the one being worked on
  const rsrc_t k_rsrc = make_rsrc(kbase, kl > 0 ? (uint32_t)(((int64_t)(kl - 1) * a.k_ss + a.D) * 4) : 0u);
  const rsrc_t v_rsrc = make_rsrc(vbase, kl > 0 ? (uint32_t)(((int64_t)(kl - 1) * fa.v_ss + a.D) * 4) : 0u);
  uint4 kreg[LOADS], vreg[LOADS];
  auto fetch = [&](int kt) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int v = tid + i * kBlock;
      const int row = v / VEC_ROW, c = v % VEC_ROW;
      const int key = kt * BK + row;
      const bool in = key < kl && c * EPV < a.D;
      kreg[i] = buffer_load16(k_rsrc, in ? (uint32_t)(((int64_t)key * a.k_ss + c * EPV) * 4) : kOutOfRange);
      vreg[i] = buffer_load16(v_rsrc, in ? (uint32_t)(((int64_t)key * fa.v_ss + c * EPV) * 4) : kOutOfRange);
    }
  };
  fetch(0);

  floatx16 o[DMT];
#pragma unroll
  for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
    for (int x = 0; x < 16; ++x) o[mt][x] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const float c_exp = fa.scale * kLog2e;

  for (int kt = 0; kt < nkt; ++kt) {
    __syncthreads();                              // every wave has left the previous tile
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int v = tid + i * kBlock;
      const int row = v / VEC_ROW, c = v % VEC_ROW;
      *reinterpret_cast<uint4 *>(&lds_k[row * KP + c * EPV]) = kreg[i];
      *reinterpret_cast<uint4 *>(&lds_v[row * VP + c * EPV]) = vreg[i];
    }
    __syncthreads();
    if (kt + 1 < nkt) fetch(kt + 1);

    const int k0 = kt * BK + wk * 32;             // first key of this wave's block
    if (k0 >= vis_max) continue;                  // wave-uniform: nothing for this wave's queries here

    // ---- S^T = K Q^T
    floatx16 s;
#pragma unroll
    for (int x = 0; x < 16; ++x) s[x] = 0.f;
#pragma unroll
    for (int vs = 0; vs < NVS; ++vs) {
      const uint4 kf = *reinterpret_cast<const uint4 *>(&lds_k[(wk * 32 + r) * KP + M::k_of(vs, g, NVS)]);
      M::step(kf, qf[vs], s);
    }

    float lo, hi;
    halves_of(softmax_f32_keys(s, o, m_run, l_run, vis_l - k0 - 4 * g, k0 + 32 <= vis_min, c_exp), lo, hi);
    l_run += lo + hi;

    // ---- O^T += V^T P^T: step (j, i) contracts over keys 8j + i (lanes 0..31) and 8j + 4 + i (lanes 32..63)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float *vrow = &lds_v[(wk * 32 + 8 * j + 4 * g) * VP + r];
      const uint4 pb = make_uint4(__float_as_uint(s[4 * j]), __float_as_uint(s[4 * j + 1]), __float_as_uint(s[4 * j + 2]),
                                  __float_as_uint(s[4 * j + 3]));
#pragma unroll
      for (int mt = 0; mt < DMT; ++mt) {
        const uint4 va = make_uint4(__float_as_uint(vrow[mt * 32]), __float_as_uint(vrow[VP + mt * 32]),
                                    __float_as_uint(vrow[2 * VP + mt * 32]), __float_as_uint(vrow[3 * VP + mt * 32]));
        M::step(va, pb, o[mt]);
      }
    }
  }

  // ---- combine the two waves of a query half (they saw disjoint keys), then normalise and store.
  // Wave (wq, 1) leaves maximum, sum and output in LDS, value by value with the lane fastest; wave (wq, 0) merges.
  __syncthreads();
  float *comb = lds_v + wq * (2 + DMT * 16) * kWave;      // 2 x 34 x 64 floats: inside the V tile's 64 x 72
  if (wk == 1) {
    comb[lane] = m_run;
    comb[kWave + lane] = l_run;
#pragma unroll
    for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
      for (int x = 0; x < 16; ++x) comb[(2 + mt * 16 + x) * kWave + lane] = o[mt][x];
  }
  __syncthreads();
  if (!NORM && wk == 1) return;
  if (wk == 0) {
    const auto [w0, w1, l, inv] = pair_weights(m_run, l_run, comb[lane], comb[kWave + lane], c_exp);
    if (!NORM && q_lane >= ql) return;
    T *crow = cbase + (int64_t)q_lane * fa.c_ss;
#pragma unroll
    for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = mt * 32 + 8 * j + 4 * g;
        float4 v;
        v.x = (o[mt][4 * j + 0] * w0 + comb[(2 + mt * 16 + 4 * j + 0) * kWave + lane] * w1) * inv;
        v.y = (o[mt][4 * j + 1] * w0 + comb[(2 + mt * 16 + 4 * j + 1) * kWave + lane] * w1) * inv;
        v.z = (o[mt][4 * j + 2] * w0 + comb[(2 + mt * 16 + 4 * j + 2) * kWave + lane] * w1) * inv;
        v.w = (o[mt][4 * j + 3] * w0 + comb[(2 + mt * 16 + 4 * j + 3) * kWave + lane] * w1) * inv;
        if constexpr (NORM) {
          *reinterpret_cast<float4 *>(&lds_k[(wq * 32 + r) * KP + d]) = v;
        } else if (d < a.D) {
          if (fa.c_vec16) *reinterpret_cast<float4 *>(crow + d) = v;
          else { crow[d] = v.x; crow[d + 1] = v.y; crow[d + 2] = v.z; crow[d + 3] = v.w; }
        }
      }
  }
  if constexpr (NORM) {
    // Out as whole rows through the K tile's LDS: the stores go past the caches, where a lane's 16-byte pieces of a row of
    // its own would each be a memory access (twelve BERT-base layers, batch 8: 190 -> 182 us).
    __syncthreads();
    const rsrc_t c_rsrc = make_rsrc(cbase, (uint32_t)(((int64_t)(ql - 1) * fa.c_ss + a.D) * 4));
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int v = tid + i * kBlock, row = v / VEC_ROW, d = v % VEC_ROW * EPV;
      buffer_store16<kAgentScope>(c_rsrc, q0 + row < ql && d < a.D ? (uint32_t)((int64_t)(q0 + row) * fa.c_ss + d) * 4u : kOutOfRange,
                                  *reinterpret_cast<const uint4 *>(&lds_k[row * KP + d]));
    }
    norm_tile<EN_F32, DP>(*norm, rows);
  }
}

template <int DP>
__global__ __launch_bounds__(kBlock) void attn_fused_f32_kernel(FusedArgs fa) { fused_f32_tile<DP, false>(fa, nullptr); }
template <int DP>
__global__ __launch_bounds__(kBlock) void attn_fused_norm_f32_kernel(FusedArgs fa, NormArgs norm) { fused_f32_tile<DP, true>(fa, &norm); }

// Heads of 65..128 channels.  A wave's share of a 64-key tile is 2 x 64 MFMAs of 64 cycles, and the loads, the softmax and the LDS reads of
// one workgroup run beside the MFMAs of the others on its CU.  The matrix cores are busy 0.55 of the time where workgroups fill them evenly
// (16 of 100..384, 20 x 80, no mask: 109 us for 45 us of products), 0.31 with rows of two tiles (22 of 110, 45 x 128: 109 us), 0.37 where
// the longest tiles end alone (2 of 375..1500, 16 x 128: 176 us, 0.87 waves a SIMD); small batches are one workgroup's chain (8 of 16..128,
// 16 x 96: 15 us, 0.11).  The same split as above (64 query rows, wave (wq, wk) takes 32 of them and 32 keys of every tile, the pair is
// combined at the end), but the tiles travel from memory straight into LDS, one buffer each for K and V: V of a tile is sent for at the
// top of its step and needed behind S^T, K of the next one behind the barrier in mid-step, when every wave has left this one's, and
// needed at the end.  64 KB (48 at 96 channels) and no registers for tiles in flight: two workgroups (three) on a CU.  Layers with the
// LayerNorm, QK^T + softmax + PV / this: 2 layers of 2 sequences of up to 1500, 16 heads x 128 281 / 188 us, 6 of 8 of up to 128, 16 x 96
// 252 / 128.
//
// Rows are DP channels without padding; chunk c (16 bytes) of a K row r sits in slot c ^ kswz(r), so that the fragment reads of
// sixteen consecutive rows at one chunk cover all banks; V is read a channel a lane, rows four keys apart in the wave's halves: with
// rows of 512 bytes every key's chunks 8..15 and 0..7 trade places for keys with bit 2 set, rows of 384 bytes lie 32 banks apart,
// and there such keys trade places with their neighbour.
template <int DP>
__global__ __launch_bounds__(kBlock, DP == 96 ? 3 : 2) void attn_fused_f32_wide_kernel(FusedArgs fa) {
  typedef float T;
  typedef Mma<EN_F32> M;
  const AttnArgs &a = fa.base;
  constexpr int EPV = 4, BK = 64, NVS = DP / M::KPV, DMT = DP / 32, CPR = DP / EPV, LOADS = BK * CPR / kBlock;
  constexpr float kLog2e = 1.4426950408889634f;
  static_assert(DP == 96 || DP == 128, "swizzles are written for 24 or 32 slots per row");
  __shared__ __attribute__((aligned(16))) float lds[2 * BK * DP];
  float *const lds_k = lds, *const lds_v = lds + BK * DP;
  constexpr int HANDED = (2 + DMT * 8) * kWave;    // what a wave hands to the other of its pair: maximum, sum and half of its channels
  static_assert(4 * HANDED <= 2 * BK * DP, "the pairs are combined in the tiles' room");
  auto kswz = [](int row) { return DP == 128 ? (row & 15) : ((row >> 1) & 7); };
  auto vflip = [](int key) { return (key >> 2) & 1; };

  const SeqAhead ahead = seq_ahead(a, fa.q_row0, fa.k_row0);
  int unit, qi;
  if (!map_block(a, unit, qi)) return;
  const int b = unit / a.H, h = unit % a.H;
  const Seq seq = seq_of(a, ahead, b, fa.q_row0, fa.k_row0);
  const int kl = seq.kl, ql = seq.ql;
  const int q0 = qi * kF32QTile;
  if (q0 >= ql) return;
  const int nk = tile_key_extent(a, min(q0 + kF32QTile, ql) - 1, kl, ql);
  const int nkt = (nk + BK - 1) / BK;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, g = lane >> 5;
  const int wq = wave & 1, wk = wave >> 1;
  const int q_first = q0 + wq * 32, q_lane = q_first + r;
  // keys this lane's query may see, and the wave's smallest and largest such extent
  const int vis_l = (q_lane < ql) ? (a.causal ? min(kl, q_lane + (kl - ql) + 1) : kl) : 0;
  const int vis_min = (q_first + 31 < ql) ? (a.causal ? min(kl, q_first + (kl - ql) + 1) : kl) : 0;
  const int vis_max = (q_first < ql) ? (a.causal ? min(kl, min(q_first + 31, ql - 1) + (kl - ql) + 1) : kl) : 0;

  const int64_t qr = seq.q_row, kr = seq.k_row;
  const T *qbase = reinterpret_cast<const T *>(a.a_ptr) + (int64_t)b * a.q_sb + qr * a.q_ss + (int64_t)h * a.q_sh;
  const T *kbase = reinterpret_cast<const T *>(a.b_ptr) + (int64_t)b * a.k_sb + kr * a.k_ss + (int64_t)h * a.k_sh;
  const T *vbase = reinterpret_cast<const T *>(fa.v) + (int64_t)b * fa.v_sb + kr * fa.v_ss + (int64_t)h * fa.v_sh;
  T *cbase = reinterpret_cast<T *>(a.out) + (int64_t)b * fa.c_sb + qr * fa.c_ss + (int64_t)h * fa.c_sh;

  // K / V tiles: the descriptors end with the last valid key, so rows past it arrive as zeros
  const desc_t k_desc = make_desc(kbase, kl > 0 ? (uint32_t)(((int64_t)(kl - 1) * a.k_ss + a.D) * 4) : 0u);
  const desc_t v_desc = make_desc(vbase, kl > 0 ? (uint32_t)(((int64_t)(kl - 1) * fa.v_ss + a.D) * 4) : 0u);
  const uint32_t k_row_bytes = (uint32_t)(a.k_ss * 4), v_row_bytes = (uint32_t)(fa.v_ss * 4);
  uint32_t k_off[LOADS], v_off[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (i * kBlock + tid) / CPR, slot = (i * kBlock + tid) % CPR;
    const int k_c = slot ^ kswz(row), v_c = DP == 128 ? slot ^ (8 * vflip(row)) : slot, v_key = DP == 128 ? row : row ^ vflip(row);
    k_off[i] = k_c * EPV < a.D ? row * k_row_bytes + k_c * 16 : kOutOfRange;
    v_off[i] = v_c * EPV < a.D ? v_key * v_row_bytes + v_c * 16 : kOutOfRange;
  }
  auto fetch = [&](const desc_t &desc, const float *dst, uint32_t (&off)[LOADS], uint32_t row_bytes) {
    const uint32_t at = lds_address(dst) + wave * kWave * 16;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      buffer_load16_to_lds(desc, at + i * kBlock * 16, off[i]);
      off[i] += BK * row_bytes;
    }
  };
  fetch(k_desc, lds_k, k_off, k_row_bytes);

  // Q fragments: this lane's query row, four channels per step (rows past the last valid one are never stored)
  uint4 qf[NVS];
  {
    const T *qrow = qbase + (int64_t)min(q_lane, ql - 1) * a.q_ss;
#pragma unroll
    for (int vs = 0; vs < NVS; ++vs) {
      const int d = M::k_of(vs, g, NVS);
      qf[vs] = (d < a.D) ? *reinterpret_cast<const uint4 *>(qrow + d) : zero4();
    }
  }

  floatx16 o[DMT];
#pragma unroll
  for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
    for (int x = 0; x < 16; ++x) o[mt][x] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const float c_exp = fa.scale * kLog2e;
  const int ksw = kswz(r);
  const float *const krow = lds_k + (wk * 32 + r) * DP;          // wk * 32 leaves the swizzle of a row alone
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();

  for (int kt = 0; kt < nkt; ++kt) {
    fetch(v_desc, lds_v, v_off, v_row_bytes);     // V tile kt: its room was in use until the barrier that ended the step before
    const int k0 = kt * BK + wk * 32;             // first key of this wave's block
    const bool live = k0 < vis_max;               // wave-uniform
    floatx16 s;
    if (live) {
      // ---- S^T = K Q^T, the fragments read a step ahead
#pragma unroll
      for (int x = 0; x < 16; ++x) s[x] = 0.f;
      uint4 kf[2];
      auto load_step = [&](int vs) { return *reinterpret_cast<const uint4 *>(krow + ((M::k_of(vs, g, NVS) / EPV) ^ ksw) * EPV); };
      kf[0] = load_step(0);
#pragma unroll
      for (int vs = 0; vs < NVS; ++vs) {
        if (vs + 1 < NVS) kf[(vs + 1) & 1] = load_step(vs + 1);
        M::step(kf[vs & 1], qf[vs], s);
      }

      // each half of the wave adds up its own keys
      l_run += softmax_f32_keys(s, o, m_run, l_run, vis_l - k0 - 4 * g, k0 + 32 <= vis_min, c_exp);
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();                                // V tile kt is there, K tile kt has been read
    fetch(k_desc, lds_k, k_off, k_row_bytes);     // K tile kt + 1 (past the end: zeros, no traffic)
    if (live) {
      // ---- O^T += V^T P^T: step (j, i) contracts over keys 8j + i (lanes 0..31) and 8j + 4 + i (lanes 32..63)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 pb = make_uint4(__float_as_uint(s[4 * j]), __float_as_uint(s[4 * j + 1]), __float_as_uint(s[4 * j + 2]),
                                    __float_as_uint(s[4 * j + 3]));
        // keys 8 j + 4 g + i: bit 2 is g
        auto v_at = [&](int i, int mt) {
          const int key = wk * 32 + 8 * j + 4 * g + i;
          return __float_as_uint(DP == 128 ? lds_v[key * DP + ((mt * 32) ^ (32 * g)) + r] : lds_v[(key ^ g) * DP + mt * 32 + r]);
        };
#pragma unroll
        for (int mt = 0; mt < DMT; ++mt) M::step(make_uint4(v_at(0, mt), v_at(1, mt), v_at(2, mt), v_at(3, mt)), pb, o[mt]);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();                                // K tile kt + 1 is there, V tile kt has been read
  }

  // ---- combine the two waves of a query half (they saw disjoint keys), then normalise and store: each hands over half of its channels and
  // finishes the others.  The quotient is refined: its rounding comes once, not in 1 / l and again in the product, which rows of a few
  // keys showed (context of 17 keys, 68 channels against float64 1.35e-7 -> 1.32e-7, of 40, 100 1.93e-7 -> 1.915e-7; QK^T, softmax and PV
  // 1.31e-7 and 1.91e-7; from 64 keys on theirs is the larger).
  float l_lo, l_hi;
  halves_of(l_run, l_lo, l_hi);
  l_run = l_lo + l_hi;
  float *const mine = lds + (2 * wq + wk) * HANDED, *const other = lds + (2 * wq + (wk ^ 1)) * HANDED;
  auto hand = [&](auto half) {
    mine[lane] = m_run;
    mine[kWave + lane] = l_run;
#pragma unroll
    for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
      for (int x = 0; x < 8; ++x) mine[(2 + mt * 8 + x) * kWave + lane] = o[mt][8 * decltype(half)::value + x];
  };
  auto finish = [&](auto half) {
    const auto [w0, w1, l, inv] = pair_weights(m_run, l_run, other[lane], other[kWave + lane], c_exp);
    T *crow = cbase + (int64_t)q_lane * fa.c_ss;
#pragma unroll
    for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int j = 2 * decltype(half)::value + jj, d = mt * 32 + 8 * j + 4 * g;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float sum = o[mt][4 * j + i] * w0 + other[(2 + mt * 8 + 4 * jj + i) * kWave + lane] * w1, quot = sum * inv;
          const float rest = fmaf(-quot, l, sum);
          v[i] = rest == rest ? fmaf(rest, inv, quot) : quot;      // a sum that is not finite stays what it is
        }
        if (d < a.D) *reinterpret_cast<float4 *>(crow + d) = make_float4(v[0], v[1], v[2], v[3]);
      }
  };
  typedef std::integral_constant<int, 0> Low;
  typedef std::integral_constant<int, 1> High;
  if (wk == 0) hand(High());
  else hand(Low());
  lds_barrier();
  if (q_lane >= ql) return;
  if (wk == 0) finish(Low());
  else finish(High());
}

static int launch_fused_f32_wide(const FusedArgs &fa, hipStream_t s) {
  const AttnArgs &a = fa.base;
  const unsigned grid = (unsigned)(ceil_div(a.units, kXcds) * kXcds * a.ntq);
  if (a.D <= 96) attn_fused_f32_wide_kernel<96><<<grid, kBlock, 0, s>>>(fa);
  else attn_fused_f32_wide_kernel<128><<<grid, kBlock, 0, s>>>(fa);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

int launch_fused_f32(FusedArgs &fa, const NormArgs *norm, hipStream_t s) {
  const AttnArgs &a = fa.base;
  if (a.units > 65535) return EN_ERR_SHAPE;
  const dim3 grid((unsigned)ceil_div(a.Sq, kF32QTile), (unsigned)a.units, 1);
  if (norm) attn_fused_norm_f32_kernel<64><<<grid, kBlock, 0, s>>>(fa, *norm);
  else attn_fused_f32_kernel<64><<<grid, kBlock, 0, s>>>(fa);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

}  // namespace en

extern "C" {

// us a layer, QK^T + softmax + PV / this, with the LayerNorm behind either: 1 prompt of 64, 12 heads x 128 28 / 18, 4 of up to 128, 8 x
// 80 39 / 21, 8 of up to 128, 16 x 96 43 / 23, 1 of 1000, 4 x 128 155 / 76, 4 of up to 512, 12 x 96 103 / 49, 22 of 110, 45 x 128 260 / 137,
// 16 of up to 384, 20 x 80, no mask 199 / 128, 4 of up to 35, 12 x 96 26 / 15, 64 of up to 20, 4 x 128 22 / 16, 1 of 17, 4 x 68 (the host's
// time) 23 / 15.  The faster form at every size: wherever it takes the heads, it is theirs.  Its context against float64, three kernels /
// this, 60 draws: 17 keys, 68 channels 1.306e-7 / 1.324e-7, 20, 128 1.504e-7 / 1.499e-7, 40, 100, no mask 2.985e-7 / 2.950e-7, 64, 128, no
// mask 3.585e-7 / 3.462e-7, 1200, 128, no mask 7.45e-7 / 6.04e-7.
int en_attn_fused_f32_wide_pays(int batch, int head_num, int max_seq_len, int size_per_head) {
  return batch > 0 && head_num > 0 && max_seq_len > 0 && size_per_head > 64 && size_per_head <= 128 && size_per_head % 4 == 0;
}

int en_attn_fused_f32_wide(const void *qkv, void *ctx, const int32_t *seq_lens, const int32_t *cu_seqlens, int batch, int head_num,
                           int max_seq_len, int size_per_head, float scale, int causal, en_stream_t stream) {
  using namespace en;
  if (!qkv || !ctx || !seq_lens || !cu_seqlens) return EN_ERR_NULL;
  if (batch < 1 || head_num < 1 || max_seq_len < 1 || size_per_head < 1) return EN_ERR_SHAPE;
  if (!en_attn_fused_f32_wide_pays(batch, head_num, max_seq_len, size_per_head) || !(scale > 0.f)) return EN_ERR_UNSUPPORTED;
  if (!aligned_to(qkv, 16) || !aligned_to(ctx, 16)) return EN_ERR_ALIGN;
  const int64_t D = size_per_head, row = (int64_t)3 * head_num * D;
  if ((int64_t)batch * head_num > INT32_MAX / 64) return EN_ERR_SHAPE;
  // 32-bit byte offsets, advanced a tile at a time up to two tiles past the end, and a grid of 32 bits
  if (((int64_t)max_seq_len + 256) * row * 4 >= (1ll << 31)) return EN_ERR_UNSUPPORTED;
  FusedArgs fa{};
  AttnArgs &a = fa.base;
  const float *pk = static_cast<const float *>(qkv);
  a.a_ptr = pk; a.b_ptr = pk + D; a.out = ctx; a.k_lens = seq_lens;
  a.B = batch; a.H = head_num; a.Sq = max_seq_len; a.Sk = max_seq_len; a.D = size_per_head;
  a.q_sh = a.k_sh = fa.v_sh = 3 * D;
  a.q_ss = a.k_ss = fa.v_ss = row;
  a.alpha = 1.f; a.causal = causal ? 1 : 0;
  a.ntq = (int)ceil_div(max_seq_len, kF32QTile);
  a.units = batch * head_num;
  fa.v = pk + 2 * D;
  fa.c_sh = D; fa.c_ss = head_num * D;
  fa.q_row0 = fa.k_row0 = cu_seqlens;
  fa.scale = scale;
  if (ceil_div(a.units, kXcds) * kXcds * a.ntq > INT32_MAX) return EN_ERR_SHAPE;
  return launch_fused_f32_wide(fa, (hipStream_t)stream);
}

}  // extern "C"
