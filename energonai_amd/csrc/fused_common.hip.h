// What the two fused attention kernels share: the argument block and two lane-level helpers.
#pragma once

#include "attn_common.hip.h"

#include <math.h>

namespace en {

// The lane's number in its wave, counted afresh (two VALU instructions) where a value derived from it is needed only
// now and then, instead of keeping that value in a register through the key loop: the kernel has none to spare.
__device__ __forceinline__ int lane_now() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

struct FusedArgs {
  AttnArgs base;             // a_ptr = q, b_ptr = k, out = ctx; q_s* = q strides, k_s* = k strides
  const void *v;
  int64_t v_sb, v_sh, v_ss;
  int64_t c_sb, c_sh, c_ss;
  const int32_t *q_row0;     // packed layout: first row of batch b in q / ctx (else null)
  const int32_t *k_row0;     // packed layout: first row of batch b in k / v (else null)
  float scale;
  int c_vec16;               // ctx rows may be written with 128-bit stores (16-byte aligned base and strides)
};

// ---- residual + LayerNorm behind the attention, in its launch -----------------------------------------------------------
// Where the LayerNorm follows the attention directly (its width is heads * size_per_head), the H workgroups of a query tile,
// one per head, wait for each other once their context rows are written, and each normalises an H-th of the tile's rows.
// That is worth it while the workgroups of a launch are all resident at once: one launch less per layer, and the residual
// rows, gamma and beta are on their way while the workgroups meet.
//
// The meeting point is one 64-bit word per (sequence, query tile), zero between launches: bits 0..5 count the workgroups
// that have arrived, bits 6..11 those that have gone on, bit 12 + h says that head h has gone without doing its rows.  No
// workgroup waits without end: after `polls` looks it sets its bit and leaves, unless the last one arrived in the meantime;
// the last to arrive finds the bits set before its own arrival and does those rows too.  So every row has exactly one owner
// in whatever order the workgroups run, and the word returns to zero when all H shares have gone on.
struct NormArgs {
  const void *residual;
  const int32_t *res_off;       // residual row of output row t is t + res_off[t]
  const void *gamma, *beta;
  const void *ctx;              // packed [T, width], written by this launch
  void *out;
  unsigned long long *arrivals; // [batch][ntq], kNormWordStride apart
  int width, polls;
  float eps;
};
// A memory channel's 256 bytes per word: neighbours in one line make all workgroups of a batch queue for it.
constexpr int kNormWordStride = 32;
constexpr int kNormMaxHeads = 48;         // shares that a meeting word has room for
constexpr int kNormMaxVectors = 4 * kWave; // a wave per row, up to four 16-byte vectors per lane
constexpr int kAgentScope = 16;           // cache policy of an access that all XCDs see (sc1)

// Rows of a wave in flight at once: the context comes from memory (other XCDs wrote it), a trip of 2 us each time otherwise.  As
// many as a wave has in most tiles and as the registers of the attention hold (head_pitch: channels of a head in LDS; at 64
// four waves share a SIMD's registers, above that three).
constexpr int norm_rows_ahead(int dt, int head_pitch, int vpl) {
  return dt == EN_F32 ? (vpl <= 3 ? 2 : 1) : vpl <= 2 ? 3 : head_pitch > 64 ? 2 : 1;
}
constexpr int kNormRowsAhead = 3;

// A workgroup's share of its tile's rows, and where the residuals of the first ones lie: scalars that are looked up before the
// keys are walked, a trip to memory less behind them.
struct NormTile {
  unsigned long long *word;
  int64_t row0;                 // packed row of the tile's first
  int nrows, share, shares;
  int res_off[kNormRowsAhead];  // of the wave's first rows
};

__device__ __forceinline__ NormTile norm_tile_of(const NormArgs &n, int64_t word, int64_t row0, int nrows, int share, int shares) {
  NormTile t{n.arrivals + word * kNormWordStride, row0, nrows, share, shares, {}};
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), step = shares * (kBlock / kWave);
#pragma unroll
  for (int k = 0; k < kNormRowsAhead; ++k)
    t.res_off[k] = n.res_off[row0 + min(share * (kBlock / kWave) + wave + k * step, nrows - 1)];
  return t;
}

template <int DT, int DP, int VPL>
__device__ __forceinline__ void norm_tile_rows(const NormArgs &n, const NormTile &t, unsigned long long *s_take) {
  unsigned long long *const word = t.word;
  const int64_t row0 = t.row0;
  const int nrows = t.nrows, share = t.share, shares = t.shares;
  typedef Elem<DT> E;
  typedef typename E::T T;
  constexpr int EPV = 16 / E::kSize, NW = kBlock / kWave;
  typedef Pack<T, EPV> P;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int nvec = n.width / EPV;
  const uint32_t bytes = (uint32_t)(n.width * E::kSize);      // the loads of vectors past the row give zeros
  constexpr bool EARLY = VPL <= 3;              // gamma and beta in registers while the workgroups meet: four vectors do not fit
  constexpr int R = norm_rows_ahead(DT, DP, VPL);
  static_assert(R <= kNormRowsAhead, "offsets looked up ahead");
  const int step = shares * NW;
  uint4 res[R][VPL];
  P g[VPL], bt[VPL];
  auto load_residual = [&](int first, auto off_of) {
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int64_t row = row0 + min(first + k * step, nrows - 1);
      const rsrc_t p = make_rsrc(reinterpret_cast<const T *>(n.residual) + (row + off_of(k, row)) * n.width,
                                 first + k * step < nrows ? bytes : 0u);
#pragma unroll
      for (int j = 0; j < VPL; ++j) res[k][j] = buffer_load16(p, (uint32_t)(lane + kWave * j) * 16u);
    }
  };
  auto load_affine = [&](int j) {
    g[j] = __builtin_bit_cast(P, buffer_load16(make_rsrc(n.gamma, bytes), (uint32_t)(lane + kWave * j) * 16u));
    bt[j] = __builtin_bit_cast(P, buffer_load16(make_rsrc(n.beta, bytes), (uint32_t)(lane + kWave * j) * 16u));
  };
  unsigned long long arrived = 0;               // what it answers comes back ahead of the loads behind it
  if (threadIdx.x == 0) {
    int at = 0;
    asm("" : "+v"(at));                         // a lane's own address: behind a uniform one the answer is waited for here and passed round
    arrived = atomicAdd(word + at, 1ull);
  }
  if constexpr (EARLY)
#pragma unroll
    for (int j = 0; j < VPL; ++j) load_affine(j);
  int held = share * NW + wave;                 // first of the rows whose residuals are in registers
  load_residual(held, [&](int k, int64_t) { return t.res_off[k]; });
  if (threadIdx.x == 0) {
    unsigned long long take = 0;                // shares to do here
    if ((int)(arrived & 63) == shares - 1) {
      take = arrived >> 12 | 1ull << share;
    } else {
      bool all = false;
      for (int i = 0; i < n.polls && !all; ++i) {
        __builtin_amdgcn_s_sleep(4);
        all = (int)(__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 63) == shares;
      }
      if (!all) all = (int)(atomicOr(word, 1ull << (12 + share)) & 63) == shares;
      if (all) take = 1ull << share;
    }
    *s_take = take;
  }
  lds_barrier();
  for (unsigned long long take = *s_take; take; take &= take - 1) {
    const int base = __builtin_amdgcn_readfirstlane((__ffsll(take) - 1) * NW + wave);
    for (int i = base; i < nrows; i += R * step) {
      uint4 raw[R][VPL];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const rsrc_t ctx = make_rsrc(reinterpret_cast<const T *>(n.ctx) + (row0 + i + k * step) * n.width,
                                     i + k * step < nrows ? bytes : 0u);
#pragma unroll
        for (int j = 0; j < VPL; ++j) raw[k][j] = buffer_load16<kAgentScope>(ctx, (uint32_t)(lane + kWave * j) * 16u);
      }
      if (i != held) load_residual(i, [&](int, int64_t row) { return __builtin_amdgcn_readfirstlane(n.res_off[row]); });
      held = i;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        __builtin_amdgcn_sched_barrier(0);      // row by row: their sums side by side take more registers than there are
        if (i + k * step >= nrows) break;
        float x[VPL][EPV], s = 0.f, d2 = 0.f;
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
          const P a = __builtin_bit_cast(P, raw[k][j]), r = __builtin_bit_cast(P, res[k][j]);
          const bool in = lane + kWave * j < nvec;
#pragma unroll
          for (int e = 0; e < EPV; ++e) {
            x[j][e] = in ? E::to_float(a.v[e]) + E::to_float(r.v[e]) : 0.f;
            s += x[j][e];
          }
        }
        const float mu = wave_allreduce<OpSum>(s) / (float)n.width;
#pragma unroll
        for (int j = 0; j < VPL; ++j)
          if (lane + kWave * j < nvec)
#pragma unroll
            for (int e = 0; e < EPV; ++e) d2 += (x[j][e] - mu) * (x[j][e] - mu);
        const float inv = 1.0f / sqrtf(wave_allreduce<OpSum>(d2) / (float)n.width + n.eps);
        T *out = reinterpret_cast<T *>(n.out) + (row0 + i + k * step) * n.width;
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
          const int v = lane + kWave * j;
          if constexpr (!EARLY) load_affine(j);
          if (v < nvec) {
            P o;
#pragma unroll
            for (int e = 0; e < EPV; ++e) {
              float f = (x[j][e] - mu) * inv * E::to_float(g[j].v[e]) + E::to_float(bt[j].v[e]);
              asm("" : "+v"(f));      // rounded to fp32 and then to the storage type, as layernorm.hip's wide rows are, not in one instruction
              o.v[e] = E::from_float(f);
            }
            store_pack<T, EPV>(out + v * EPV, o);
          }
        }
      }
    }
  }
  // off the way of the rows: the shares done here have gone on, and the last of them leaves the word at zero
  if (threadIdx.x == 0 && *s_take) {
    const int mine = __popcll(*s_take);
    const int before = (int)(atomicAdd(word, (unsigned long long)mine << 6) >> 6 & 63);
    if (before + mine == shares) __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Called by the whole workgroup when it has sent its context rows away with agent-scope stores.
template <int DT, int DP>
__device__ __forceinline__ void norm_tile(const NormArgs &n, const NormTile &t) {
  __shared__ unsigned long long s_take;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the wave's context rows are where every XCD sees them ...
  lds_barrier();                                        // ... and the other waves' too, before the workgroup says so
  const int nvec = n.width / (16 / Elem<DT>::kSize);
  if (nvec <= 2 * kWave) norm_tile_rows<DT, DP, 2>(n, t, &s_take);
  else if (nvec <= 3 * kWave) norm_tile_rows<DT, DP, 3>(n, t, &s_take);
  else norm_tile_rows<DT, DP, 4>(n, t, &s_take);
}

// Both halves of the wave get (x of lanes 0..31, x of lanes 32..63): one VALU swap, no LDS round trip.
__device__ __forceinline__ void halves_of(float x, float &lo, float &hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}

// fused_wide.hip: the kernel whose waves own 64 queries each (256-query workgroups), for heads of 65..128 channels.
constexpr int kWideQTile = 256;
int launch_fused_wide(int dtype, FusedArgs &fa, hipStream_t s);
// fused_f32.hip: fp32 storage, heads of up to 64 channels, 64-row query tiles.
int launch_fused_f32(FusedArgs &fa, const NormArgs *norm, hipStream_t s);
constexpr int kF32QTile = 64;

}  // namespace en
