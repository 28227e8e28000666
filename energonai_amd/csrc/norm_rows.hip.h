// Residual + LayerNorm as a role that some workgroups of an attention launch take: rows of [rows, width] in 16-bit storage,
//
//   out[t] = LayerNorm(in[t] + residual[t + res_off[t]]) * gamma + beta
//
// with fp32 statistics from registers and one rounding at the store, as the kernels of layernorm.hip.  A workgroup of the
// attention kernels is 256 lanes, so a row is a wave's (up to 1536 channels, four rows a workgroup and no barrier) or the
// whole workgroup's.  One row each: workgroups that go on to further rows, with the next one's loads in flight, start as many
// fewer waves and measure slower (rows of 8192 beside 16 heads x 64, 3569 tokens: one row 44 us, two 47, four 51).
#pragma once

#include "common.hip.h"

#include <math.h>

namespace en {

struct NormRows {
  const void *in, *residual;
  const int32_t *res_off;       // residual row of output row t is t + res_off[t] (null: t)
  const void *gamma, *beta;
  void *out;
  int64_t rows;
  int width;
  float eps;
  int groups;                   // workgroups of this role, in groups of one per XCD
  uint32_t step;                // of every 2^16 groups of the launch this many are of this role, until all are
};

constexpr int kNormRowsMaxVectors = 6 * kBlock;      // 16-byte vectors of a row: 12288 channels
constexpr int norm_rows_per_workgroup(int width) { return width / 8 <= 3 * kWave ? kBlock / kWave : 1; }

// TPR lanes a row (a wave or the workgroup), VPL vectors a lane.
template <int DT, int TPR, int VPL, bool STREAM>
__device__ __forceinline__ void norm_row(const NormRows &n, int64_t row) {
  typedef Elem<DT> E;
  typedef typename E::T T;
  constexpr int EPV = 8, NW = TPR / kWave, AUX = STREAM ? 2 : 0;
  typedef Pack<T, EPV> P;
  __shared__ float s_part[2][NW];
  const int t = threadIdx.x % TPR, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  // uniform over the wave; the loads of vectors past the row give zeros
  const uint32_t bytes = (uint32_t)n.width * E::kSize;
  const int64_t res_row = row + (n.res_off ? n.res_off[row] : 0);
  const rsrc_t in = make_rsrc(static_cast<const T *>(n.in) + row * n.width, bytes);
  const rsrc_t res = make_rsrc(static_cast<const T *>(n.residual) + res_row * n.width, bytes);
  const rsrc_t gamma = make_rsrc(n.gamma, bytes), beta = make_rsrc(n.beta, bytes);
  uint4 raw[VPL], rraw[VPL], g[VPL], bt[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) raw[j] = buffer_load16<AUX>(in, (uint32_t)(t + TPR * j) * 16u);
#pragma unroll
  for (int j = 0; j < VPL; ++j) rraw[j] = buffer_load16<AUX>(res, (uint32_t)(t + TPR * j) * 16u);
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    g[j] = buffer_load16(gamma, (uint32_t)(t + TPR * j) * 16u);
    bt[j] = buffer_load16(beta, (uint32_t)(t + TPR * j) * 16u);
  }
  auto row_sum = [&](float v, float *part) {
    v = wave_allreduce<OpSum>(v);
    if constexpr (NW > 1) {
      if (threadIdx.x % kWave == 0) part[wave] = v;
      lds_barrier();
      v = part[0];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += part[w];
    }
    return v;
  };
  float x[VPL][EPV], s = 0.f, d2 = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const P a = __builtin_bit_cast(P, raw[j]), r = __builtin_bit_cast(P, rraw[j]);
#pragma unroll
    for (int e = 0; e < EPV; ++e) {
      x[j][e] = E::to_float(a.v[e]) + E::to_float(r.v[e]);
      s += x[j][e];
    }
  }
  const float mu = row_sum(s, s_part[0]) / (float)n.width;
#pragma unroll
  for (int j = 0; j < VPL; ++j)
    if (t + TPR * j < n.width / EPV)
#pragma unroll
      for (int e = 0; e < EPV; ++e) d2 += (x[j][e] - mu) * (x[j][e] - mu);
  const float inv = 1.0f / sqrtf(row_sum(d2, s_part[1]) / (float)n.width + n.eps);
  const rsrc_t out = make_rsrc(static_cast<T *>(n.out) + row * n.width, bytes);
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const P gp = __builtin_bit_cast(P, g[j]), bp = __builtin_bit_cast(P, bt[j]);
    P o;
#pragma unroll
    for (int e = 0; e < EPV; ++e) {
      float f = (x[j][e] - mu) * inv * E::to_float(gp.v[e]) + E::to_float(bp.v[e]);
      asm("" : "+v"(f));      // rounded to fp32 and then to the storage type, not in one instruction
      o.v[e] = E::from_float(f);
    }
    buffer_store16<AUX>(out, (uint32_t)(t + TPR * j) * 16u, __builtin_bit_cast(uint4, o));
  }
}

// Workgroup `index` of the role.
template <int DT, bool STREAM>
__device__ __forceinline__ void norm_rows(const NormRows &n, int index) {
  const int nvec = n.width / 8;
  const int64_t row = nvec <= 3 * kWave ? (int64_t)index * (kBlock / kWave) + __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave) : index;
  if (row >= n.rows) return;
  if (nvec <= kWave) norm_row<DT, kWave, 1, STREAM>(n, row);
  else if (nvec <= 3 * kWave) norm_row<DT, kWave, 3, STREAM>(n, row);
  else if (nvec <= 2 * kBlock) norm_row<DT, kBlock, 2, STREAM>(n, row);
  else if (nvec <= 4 * kBlock) norm_row<DT, kBlock, 4, STREAM>(n, row);
  else norm_row<DT, kBlock, 6, STREAM>(n, row);
}

}  // namespace en
