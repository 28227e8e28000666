// LayerNorm forward with an optional fused residual add.
//
// Single pass over HBM: each row is read once into VGPRs with 128-bit loads
// (TPR lanes share a row, VPL vectors per lane), the mean and then the
// centred sum of squares are reduced from the registers (two-pass statistics
// without a second trip to memory: wave64 DPP reductions, LDS only to combine
// waves), and the normalised row is written once.  All arithmetic is fp32 with
// a single rounding at the store.  Rows that do not fit the register tiling,
// or are not 16-byte aligned, take the three-pass workgroup-per-row kernel.
#include "common.hip.h"

#include <math.h>

namespace en {

struct LnArgs {
  void *out;
  float *mean;
  float *invvar;
  void *sum_out;
  const void *in;
  const void *residual;
  const int32_t *res_off;   // residual row of output row t is t + res_off[t] (null: t)
  const void *gamma;
  const void *beta;
  int64_t n1;
  int n2;
  float eps;
};

// One wave per row: four rows share a workgroup and no barrier; else a workgroup is a row.
constexpr int rows_block(int tpr) { return tpr == kWave ? kBlock : tpr; }

// STREAM, STREAM_LD: the output, and the inputs, pass by the memory-side cache with non-temporal accesses (see launch_rows).
template <int DTI, int DTO, int VPL, int TPR, bool STREAM, bool STREAM_LD>
__global__ __launch_bounds__(rows_block(TPR)) void layernorm_rows_kernel(LnArgs a) {
  typedef Elem<DTI> EI;
  typedef Elem<DTO> EO;
  typedef typename EI::T TI;
  typedef typename EO::T TO;
  constexpr int BLOCK = rows_block(TPR);
  constexpr int EPV = 16 / EI::kSize;  // elements per 128-bit input vector
  constexpr int NW = TPR / kWave;      // waves sharing a row
  constexpr int ROWS_PER_BLOCK = BLOCK / TPR;
  __shared__ float s_a[NW > 1 ? NW : 1];
  __shared__ float s_b[NW > 1 ? NW : 1];

  const int t = threadIdx.x % TPR;
  const int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + threadIdx.x / TPR;
  const bool active = row < a.n1;  // uniform per wave (TPR is a multiple of 64)
  if (!active) return;             // ROWS_PER_BLOCK > 1 only when a row is one wave: no barrier follows

  const int nvec = a.n2 / EPV;
  const TI *in = reinterpret_cast<const TI *>(a.in) + row * a.n2;
  TI *sum_out = a.sum_out ? reinterpret_cast<TI *>(a.sum_out) + row * a.n2 : nullptr;

  // Rows that come out of a cache are bound by the length of their chain, so everything they need is sent for before the
  // first reduction waits for anything: gamma and beta behind the reductions would be a second trip (in a layer, 8300
  // rows of 768 fp16 9.3 -> 8.6 us, 5000 rows of 1024 bf16 7.9 -> 7.4 us; alone, 64 rows of 9216 4.5 -> 3.9 us).  Rows
  // streamed from memory are bound by what is in flight, and the registers that hold gamma and beta cost waves: there
  // they are loaded where they are used (14213 rows of 12288 fp16 166 us against 180; 9304 of 7168 67 against 70).
  // The row's own loads go out first: where the residual row is found through res_off, its address hangs on a load of
  // its own.
  // That takes registers, and past 64 of them a CU holds one workgroup of 1024 lanes instead of two, or three of 512 instead
  // of four; rows of up to three vectors on up to 512 lanes are worth it.  1000 rows, without / with residual, all sent for
  // early against a vector's operands where it is used: 16384 fp32 (1024 x 4) 26.2 / 34.1 against 21.3 / 31.2 us, 32768 fp16
  // 27.3 / 36.6 against 21.3 / 32.0, 7168 fp32 (512 x 4) 11.4 / 14.5 against 10.0 / 14.6.
  constexpr int HELD = VPL * (EPV + 4 + EPV * EO::kSize / 2);       // the row in fp32, residual, gamma and beta
  constexpr bool AHEAD = HELD <= 48 || (VPL <= 3 && TPR <= 512);
  constexpr bool EARLY = AHEAD && !STREAM;
  // The residual alone is sent for ahead on 512 lanes (2000 rows of 7168 fp32 28.2 -> 25.9 us), and where one workgroup of
  // 1024 is all that fits and has the room (1000 rows of 49152 fp16 63.4 -> 60 us; 65536 would spill).
  constexpr bool RES_AHEAD = AHEAD || TPR <= 512 || (VPL * EPV > 32 && VPL * (EPV + 8) <= 96);
  uint4 raw[VPL], rraw[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = t + TPR * j;
    raw[j] = (v < nvec) ? load16<STREAM_LD>(in + v * EPV) : make_uint4(0u, 0u, 0u, 0u);
  }
  const TO *gamma = reinterpret_cast<const TO *>(a.gamma);
  const TO *beta = reinterpret_cast<const TO *>(a.beta);
  Pack<TO, EPV> g[VPL], bt[VPL];
  auto load_affine = [&](int j) {
    const int v = min(t + TPR * j, nvec - 1);
    g[j] = load_pack<TO, EPV>(gamma + v * EPV);
    bt[j] = load_pack<TO, EPV>(beta + v * EPV);
  };
  const TI *res = a.residual ? reinterpret_cast<const TI *>(a.residual) + (row + (a.res_off ? a.res_off[row] : 0)) * a.n2 : nullptr;
  if constexpr (EARLY)
#pragma unroll
    for (int j = 0; j < VPL; ++j) load_affine(j);
  if (RES_AHEAD && res) {
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int v = t + TPR * j;
      rraw[j] = (v < nvec) ? load16<STREAM_LD>(res + v * EPV) : make_uint4(0u, 0u, 0u, 0u);
    }
  }

  float x[VPL][EPV];
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = t + TPR * j;
    if (v < nvec) {
      const Pack<TI, EPV> pk = __builtin_bit_cast(Pack<TI, EPV>, raw[j]);
#pragma unroll
      for (int e = 0; e < EPV; ++e) x[j][e] = EI::to_float(pk.v[e]);
      if (res) {
        const Pack<TI, EPV> rk = __builtin_bit_cast(Pack<TI, EPV>, RES_AHEAD ? rraw[j] : load16<STREAM_LD>(res + v * EPV));
#pragma unroll
        for (int e = 0; e < EPV; ++e) x[j][e] += EI::to_float(rk.v[e]);
      }
      if (sum_out) {
        Pack<TI, EPV> sk;
#pragma unroll
        for (int e = 0; e < EPV; ++e) sk.v[e] = EI::from_float(x[j][e]);
        store_pack<TI, EPV>(sum_out + v * EPV, sk);
      }
#pragma unroll
      for (int e = 0; e < EPV; ++e) s += x[j][e];
    } else {
#pragma unroll
      for (int e = 0; e < EPV; ++e) x[j][e] = 0.f;
    }
  }
  s = block_allreduce<OpSum, NW>(s, s_a);
  const float mu = s / (float)a.n2;
  float d2 = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = t + TPR * j;
    if (v < nvec) {
#pragma unroll
      for (int e = 0; e < EPV; ++e) {
        const float d = x[j][e] - mu;
        d2 += d * d;
      }
    }
  }
  d2 = block_allreduce<OpSum, NW>(d2, s_b);
  const float var = d2 / (float)a.n2;
  const float inv = 1.0f / sqrtf(var + a.eps);

  if constexpr (AHEAD && !EARLY)
#pragma unroll
    for (int j = 0; j < VPL; ++j) load_affine(j);
  TO *out = reinterpret_cast<TO *>(a.out) + row * a.n2;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int v = t + TPR * j;
    if (v < nvec) {
      if constexpr (!AHEAD) load_affine(j);
      Pack<TO, EPV> o;
#pragma unroll
      for (int e = 0; e < EPV; ++e)
        o.v[e] = EO::from_float((x[j][e] - mu) * inv * EO::to_float(g[j].v[e]) + EO::to_float(bt[j].v[e]));
      if constexpr (sizeof(TO) * EPV == 16) store16<STREAM>(out + v * EPV, __builtin_bit_cast(uint4, o));
      else store_pack<TO, EPV>(out + v * EPV, o);
    }
  }
  if (t == 0) {
    if (a.mean) a.mean[row] = mu;
    if (a.invvar) a.invvar[row] = inv;
  }
}

// Any n2, any alignment: one workgroup per row, three strided passes.
template <int DTI, int DTO>
__global__ __launch_bounds__(kBlock) void layernorm_generic_kernel(LnArgs a) {
  typedef Elem<DTI> EI;
  typedef Elem<DTO> EO;
  typedef typename EI::T TI;
  typedef typename EO::T TO;
  __shared__ float s_a[kBlock / kWave];
  __shared__ float s_b[kBlock / kWave];
  const int64_t row = blockIdx.x;
  const TI *in = reinterpret_cast<const TI *>(a.in) + row * a.n2;
  const TI *res = a.residual ? reinterpret_cast<const TI *>(a.residual) + (row + (a.res_off ? a.res_off[row] : 0)) * a.n2 : nullptr;
  TI *sum_out = a.sum_out ? reinterpret_cast<TI *>(a.sum_out) + row * a.n2 : nullptr;
  float s = 0.f;
  for (int i = threadIdx.x; i < a.n2; i += kBlock) {
    float v = EI::to_float(in[i]);
    if (res) v += EI::to_float(res[i]);
    s += v;
  }
  s = block_allreduce<OpSum, kBlock / kWave>(s, s_a);
  const float mu = s / (float)a.n2;
  float d2 = 0.f;
  for (int i = threadIdx.x; i < a.n2; i += kBlock) {
    float v = EI::to_float(in[i]);
    if (res) v += EI::to_float(res[i]);
    d2 += (v - mu) * (v - mu);
  }
  d2 = block_allreduce<OpSum, kBlock / kWave>(d2, s_b);
  const float inv = 1.0f / sqrtf(d2 / (float)a.n2 + a.eps);
  const TO *gamma = reinterpret_cast<const TO *>(a.gamma);
  const TO *beta = reinterpret_cast<const TO *>(a.beta);
  TO *out = reinterpret_cast<TO *>(a.out) + row * a.n2;
  for (int i = threadIdx.x; i < a.n2; i += kBlock) {
    float v = EI::to_float(in[i]);
    if (res) v += EI::to_float(res[i]);
    if (sum_out) sum_out[i] = EI::from_float(v);
    out[i] = EO::from_float((v - mu) * inv * EO::to_float(gamma[i]) + EO::to_float(beta[i]));
  }
  if (threadIdx.x == 0) {
    if (a.mean) a.mean[row] = mu;
    if (a.invvar) a.invvar[row] = inv;
  }
}

template <int DTI, int DTO, int VPL, int TPR>
static void launch_rows(const LnArgs &a, hipStream_t s) {
  constexpr int BLOCK = rows_block(TPR);
  constexpr int ROWS_PER_BLOCK = BLOCK / TPR;
  const unsigned grid = (unsigned)ceil_div(a.n1, ROWS_PER_BLOCK);
  // From kStreamStoreBytes on the output does not stay in the memory-side cache, and is stored past it.  The inputs are read out
  // of that cache where they fit it, beside what the kernel that produced them read: both together, and one of them three
  // quarters of it.  Cached / non-temporal loads, us, the input just written by a copy (and, in brackets, read again and
  // again): 6000 rows of 9216 fp16 with residual, 222 MB, 53.6 / 54.9 (49.4 / 56.1), without 35.8 / 36.1 (34.5 / 41.5); 9304 of
  // 7168 with residual, 267 MB, 63.4 / 63.8 (58.6 / 66.9); 8000 of 9216 with residual, 295 MB, 76.6 / 69.9 (73.5 / 73.5);
  // 2000 of 49152 without, 197 MB, 77.1 / 74.3 (69.9 / 79.5), 9000 of 12288, 221 MB, 78.1 / 70.2 (64.6 / 75.5).
  const int64_t elems = a.n1 * a.n2, bytes = elems * Elem<DTO>::kSize, in = elems * Elem<DTI>::kSize;
  const bool fits = in * (a.residual ? 2 : 1) <= kMemorySideCache && in <= kMemorySideCache / 4 * 3;
  if (bytes >= kStreamStoreBytes && !fits) layernorm_rows_kernel<DTI, DTO, VPL, TPR, true, true><<<grid, BLOCK, 0, s>>>(a);
  else if (bytes >= kStreamStoreBytes) layernorm_rows_kernel<DTI, DTO, VPL, TPR, true, false><<<grid, BLOCK, 0, s>>>(a);
  else layernorm_rows_kernel<DTI, DTO, VPL, TPR, false, false><<<grid, BLOCK, 0, s>>>(a);
}

// Launches the instance with the fewest of VPLS vectors per lane that cover the row.
template <int DTI, int DTO, int TPR, int VPL, int... MORE>
static bool launch_vpl(const LnArgs &a, int nvec, hipStream_t s) {
  if (nvec <= VPL * TPR) {
    launch_rows<DTI, DTO, VPL, TPR>(a, s);
    return true;
  }
  if constexpr (sizeof...(MORE) > 0) return launch_vpl<DTI, DTO, TPR, MORE...>(a, nvec, s);
  return false;
}

template <int DTI, int DTO>
static int dispatch(const LnArgs &a, hipStream_t s) {
  constexpr int EPV = 16 / Elem<DTI>::kSize;
  constexpr int OUT_VEC_BYTES = EPV * Elem<DTO>::kSize;
  if (a.n1 > (int64_t)INT32_MAX) return EN_ERR_SHAPE;
  const bool vec_ok = (a.n2 % EPV) == 0 && aligned_to(a.in, 16) && aligned_to(a.out, OUT_VEC_BYTES) &&
                      aligned_to(a.gamma, OUT_VEC_BYTES) && aligned_to(a.beta, OUT_VEC_BYTES) &&
                      (!a.residual || aligned_to(a.residual, 16)) && (!a.sum_out || aligned_to(a.sum_out, 16));
  const int nvec = vec_ok ? a.n2 / EPV : 0;
  bool done = false;
  if (vec_ok) {
    // Lanes per row, measured for widths of 768..12288 fp16 (96..1536 vectors) at a few hundred and at thousands of rows:
    // one wave per row (no barrier) up to three vectors per lane (1536-wide x 6000: 9.7 us, 128 x 2 10.4, 256 x 1 11.0;
    // 1600-wide x 5400: 64 x 4 13.9, 128 x 2 12.8); then two vectors per lane on 128 lanes, three where they fit
    // (3072-wide x 4000: 128 x 3 12.4, 256 x 2 13.0; 4096-wide: 128 x 4 18.1, 256 x 2 18.1, and 3.8 against 3.7 at 300 rows),
    // 256 lanes up to three (5120-wide x 3000: 17.4, 512 x 2 18.0), 512 up to four (7168-wide x 3000: 512 x 2 26.3, 256 x 4
    // 26.8; 12288-wide x 12410: 512 x 3 152.7, 256 x 6 157.6, 1024 x 2 153.3)
    done = launch_vpl<DTI, DTO, 64, 1, 2, 3>(a, nvec, s) || launch_vpl<DTI, DTO, 128, 2, 3>(a, nvec, s) ||
           launch_vpl<DTI, DTO, 256, 2, 3>(a, nvec, s) || launch_vpl<DTI, DTO, 512, 2, 3, 4>(a, nvec, s) ||
           launch_vpl<DTI, DTO, 1024, 3, 4, 6, 8>(a, nvec, s);
  }
  if (!done) layernorm_generic_kernel<DTI, DTO><<<(unsigned)a.n1, kBlock, 0, s>>>(a);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

}  // namespace en

extern "C" int en_layernorm_fwd(void *out, float *mean, float *invvar, void *sum_out, const void *in,
                                const void *residual, const int32_t *residual_row_offsets, const void *gamma,
                                const void *beta, int64_t n1, int64_t n2, float eps, int in_dtype, int out_dtype,
                                en_stream_t stream) {
  using namespace en;
  if (!out || !in || !gamma || !beta) return EN_ERR_NULL;
  if (n1 < 0 || n2 < 1 || n2 > (int64_t)INT32_MAX) return EN_ERR_SHAPE;
  if (n1 == 0) return EN_OK;
  const int esi = dtype_size(in_dtype), eso = dtype_size(out_dtype);
  if (!esi || !eso) return EN_ERR_DTYPE;
  if (!aligned_to(in, esi) || !aligned_to(out, eso) || !aligned_to(gamma, eso) || !aligned_to(beta, eso) ||
      (residual && !aligned_to(residual, esi)) || (sum_out && !aligned_to(sum_out, esi)))
    return EN_ERR_ALIGN;
  if (residual_row_offsets && !residual) return EN_ERR_NULL;
  LnArgs a{out, mean, invvar, sum_out, in, residual, residual_row_offsets, gamma, beta, n1, (int)n2, eps};
  hipStream_t s = (hipStream_t)stream;
  if (in_dtype == EN_F32 && out_dtype == EN_F32) return dispatch<EN_F32, EN_F32>(a, s);
  if (in_dtype == EN_F32 && out_dtype == EN_F16) return dispatch<EN_F32, EN_F16>(a, s);
  if (in_dtype == EN_F32 && out_dtype == EN_BF16) return dispatch<EN_F32, EN_BF16>(a, s);
  if (in_dtype == EN_F16 && out_dtype == EN_F16) return dispatch<EN_F16, EN_F16>(a, s);
  if (in_dtype == EN_BF16 && out_dtype == EN_BF16) return dispatch<EN_BF16, EN_BF16>(a, s);
  return EN_ERR_DTYPE;
}
