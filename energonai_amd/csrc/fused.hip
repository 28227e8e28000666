// Fused attention for the padded [B,H,S,*] layout and for the packed layout
// (all valid tokens back to back, no padding rows anywhere):
//
//   ctx = softmax(scale * Q K^T, causal / key-padding mask) V
//
// in one kernel, so the [B,H,Sq,Sk] score tensor never exists in HBM.  This is
// an addition to the reference's API (its callers run matmul, softmax, matmul,
// examples/bert/bert.py:108-119); the three separate ops stay available.
//
// Workgroup: 4 waves, one tile of 128 query rows of one (batch, head); wave w
// owns query rows 32w..32w+31 and every channel.  Per 64-key tile:
//
//   S^T = K Q^T      A = K rows from LDS, B = Q fragments held in registers.
//                    The 32x32 result gives each lane ONE query (its column)
//                    and 16 of the 32 keys, so row maxima and sums are
//                    per-lane reductions plus one exchange between the two
//                    lane groups.
//   online softmax   running max / sum per lane; exp2 with the scale folded in.
//   O^T += V^T P^T   A = V^T, read out of the row-major V tile with the LDS
//                    transposing read (four keys of one channel per lane and
//                    instruction), B = the probabilities straight out of the
//                    S^T accumulators, rounded to the storage type: a lane's
//                    registers (j, i) hold keys 8j + 4g + i, and the A operand
//                    simply reads V at those same keys, so P never touches LDS.
//
// K/V tiles travel from memory straight into LDS (bounds-checked loads that
// write LDS): no registers hold a tile in flight and no instruction copies
// one.  Rows keep their 16-byte chunks in XOR-swizzled slots so that both kinds
// of fragment read are free of bank conflicts.  Rows of up to 96 channels: K and V have two buffers each and are
// a tile ahead, one barrier per tile (24 sequences of up to 384 keys, 16 heads x 64, non-causal, eight layers:
// 274 -> 267 us against one V buffer; 48 KB of LDS at 96 channels is the same three workgroups per CU either way, and
// a fourth one would need 128 registers: 28 bytes of scratch, 69 -> 88 us).  Rows of 128 channels: K has two buffers, V
// one, sent for at the top of its own tile to arrive behind the score and softmax work: 48 KB of LDS, so that three
// workgroups fit a CU.  The barriers order LDS only, as in the unfused kernels.
//
// Heads of 65..96 channels have rows of 12 slots of their own instead of the 128-channel form's 16: three quarters of
// the tile loads and LDS, 22 (up to 80 channels) or 24 MFMAs per wave and tile instead of 32, and registers for the
// second V buffer.  7 sequences of up to 1531 keys, 20 heads x 80, bf16: 80.2 -> 69.1 us.
//
// Everything that crosses the memory interface does so as whole rows: the K and
// V tiles, the workgroup's Q rows (loaded straight into the buffers that are
// idle before the key loop, each lane then reads its fragments from LDS) and the
// output tile (written to the K buffers behind the loop's last barrier, stored
// 16 bytes per lane).  A lane that fetches or stores pieces of a row of its own
// makes every instruction touch 32 rows, and the queue of the address unit then
// stands full and holds back the tile loads of every wave on the CU.
#include "fused_common.hip.h"
#include "norm_rows.hip.h"

#include <algorithm>

namespace en {

// DP: channels of a row in LDS (the head size rounded up to 64, 96 or 128); NVS: MFMA steps of 16 channels that hold any.
// NORM: the residual + LayerNorm of fused_common.hip.h follows (16-byte context rows, no separate query lengths).  Q_ONCE: Q is read
// non-temporal (a parameter: chosen by a branch in the kernel, it cost the key loop registers and layers of 128 channels 10 %).
template <int DT, int DP, int NVS, bool NORM, bool Q_ONCE>
__device__ __forceinline__ void fused_tile(const FusedArgs &fa, const NormArgs *norm, int bid = blockIdx.x) {
  static_assert(DT != EN_F32, "the fused kernel is built for 16-bit storage");
  typedef Elem<DT> E;
  typedef typename E::T T;
  typedef Mma<DT> M;
  const AttnArgs &a = fa.base;
  constexpr int EPV = 8;
  constexpr int BK = 64;                         // keys per tile
  constexpr int KB = BK / 32;                    // 32-key MFMA blocks per tile
  constexpr int DMT = DP / 32;                   // 32-channel MFMA tiles of the output
  constexpr int ROW = DP;                        // LDS pitch of a K or V row: tiles are written by direct loads, unpadded
  constexpr int KVEC_ROW = DP / EPV;             // 16-byte slots per row
  constexpr int KLOADS = BK * KVEC_ROW / kBlock; // direct-load instructions per wave and tile, for each of K and V
  constexpr float kLog2e = 1.4426950408889634f;
  constexpr int NVB = DP <= 96 ? 2 : 1;          // V buffers
  static_assert(DP == 64 || DP == 96 || DP == 128, "swizzles are written for 8, 12 or 16 slots per row");
  static_assert(NVS * 16 <= DP, "a step reads channels the tile has");
  static_assert(BK * KVEC_ROW % kBlock == 0 && 32 * KVEC_ROW % kWave == 0, "tiles must divide over the block");
  __shared__ __attribute__((aligned(16))) T lds_k[2][BK * ROW];
  __shared__ __attribute__((aligned(16))) T lds_v[NVB][BK * ROW];
  // chunk held by slot c of row r: c ^ kswz(r) in a K tile (and in the staged Q rows), c ^ vswz(r) in a V tile
  auto kswz = [](int row) { return DP == 128 ? (row & 15) : DP == 96 ? ((row >> 2) & 3) : ((row >> 1) & 7); };
  auto vswz = [](int row) { return DP == 128 ? 4 * (row & 3) : DP == 96 ? 0 : 4 * ((row >> 1) & 1); };

  const SeqAhead ahead = seq_ahead(a, fa.q_row0, fa.k_row0);
  int unit, qi;
  if (!map_block(a, unit, qi, bid)) return;
  const int b = unit / a.H, h = unit % a.H;
  const Seq seq = seq_of(a, ahead, b, fa.q_row0, fa.k_row0);
  const int kl = seq.kl, ql = seq.ql;
  // The query tiles of a sequence are laid from its END: tile i of n covers rows ql - (n - i) * 128 .. and the ragged
  // tile is the first one (rows below 0 do not exist), whose walk over the keys is the shortest under a causal mask.
  // Laid from the start, the ragged tile would be the last one: a few rows holding a slot for the longest walk.
  const int ntl = (ql + kQTile - 1) / kQTile;
  if (qi >= ntl) return;
  const int q0 = ql - (ntl - qi) * kQTile;
  const int nk = tile_key_extent(a, min(q0 + kQTile, ql) - 1, kl, ql);
  const int nkt = (nk + BK - 1) / BK;
  NormTile rows;
  if constexpr (NORM)
    rows = norm_tile_of(*norm, (int64_t)b * a.ntq + qi, seq.q_row + max(q0, 0), min(q0 + kQTile, ql) - max(q0, 0), h, a.H);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, g = lane >> 5;
  // smallest and largest extent among the wave's 32 queries (wave-uniform): tiles below the
  // smallest need no masking, tiles from the largest on hold nothing for this wave
  const int q_first = q0 + wave * 32;
  const int vis_min = (q_first + 31 < ql) ? (a.causal ? min(kl, q_first + (kl - ql) + 1) : kl) : 0;
  const int vis_max = (q_first < ql && q_first + 31 >= 0) ? (a.causal ? min(kl, min(q_first + 31, ql - 1) + (kl - ql) + 1) : kl) : 0;

  // batch base: b * batch stride (padded layout) or first-row * row stride (packed layout)
  const int64_t qr = seq.q_row, kr = seq.k_row;
  const T *qbase = reinterpret_cast<const T *>(a.a_ptr) + (int64_t)b * a.q_sb + qr * a.q_ss + (int64_t)h * a.q_sh;
  const T *kbase = reinterpret_cast<const T *>(a.b_ptr) + (int64_t)b * a.k_sb + kr * a.k_ss + (int64_t)h * a.k_sh;
  const T *vbase = reinterpret_cast<const T *>(fa.v) + (int64_t)b * fa.v_sb + kr * fa.v_ss + (int64_t)h * fa.v_sh;
  T *cbase = reinterpret_cast<T *>(a.out) + (int64_t)b * fa.c_sb + qr * fa.c_ss + (int64_t)h * fa.c_sh;

  // Q fragments (B operand of S^T = K Q^T): this lane's query row, 8 channels per step.  The wave's 32 rows come in
  // as whole rows, memory straight into LDS (the second K buffer and the V buffer are idle until the key loop starts;
  // waves 0 and 1 take the one, waves 2 and 3 the other, 32 rows each), chunks in the K tile's swizzled slots, and
  // each lane then reads its own row's chunks: sixteen-byte pieces fetched by every lane from a row of its own
  // kept the address unit busy with 32 rows per instruction.
  uint4 qf[NVS];
  T *q_stage = (wave < 2 ? lds_k[1] : lds_v[NVB - 1]) + (wave & 1) * 32 * ROW;
  {
    const desc_t q_desc = make_desc(qbase, (uint32_t)(((int64_t)(ql - 1) * a.q_ss + a.D) * E::kSize));
#pragma unroll
    for (int n = 0; n < 32 * KVEC_ROW / kWave; ++n) {
      const int rr = (n * kWave + lane) / KVEC_ROW, slot = (n * kWave + lane) % KVEC_ROW;   // row of the wave's 32
      const int c = slot ^ kswz(rr);
      const int qq = q0 + wave * 32 + rr;
      const uint32_t off = (uint32_t)(((int64_t)qq * a.q_ss + c * EPV) * E::kSize);
      buffer_load16_to_lds<Q_ONCE ? 2 : 0>(q_desc, lds_address(q_stage) + n * kWave * 16, ((unsigned)qq < (unsigned)ql && c * EPV < a.D) ? off : kOutOfRange);
    }
  }

  // K / V tiles: the descriptors end with the last valid key, so rows past it (and whole tiles past the last
  // one) arrive as zeros with no traffic and no branches.  One direct load of a wave fills 1 KB of LDS, lane i
  // the 16 bytes at 16 i: the tile's slots in order, 64 of them from slot 256 n + 64 wave on for the wave's n-th load.
  // Which 16-byte chunk of the row a slot holds is the lane's choice of offset:
  //   K: slot c of row r holds chunk c ^ kswz(r), kswz = r & 15 (16 slots), (r >> 2) & 3 (12 slots: rows lie 48 banks
  //      apart, so every fourth row starts at the same bank) or (r >> 1) & 7 (8 slots): the 128-bit fragment reads of
  //      16 consecutive rows at one chunk then cover all 64 banks once;
  //   V: slot c of key k holds chunk c ^ vswz(k), vswz = 4 (k & 3) (16 slots), 0 (12 slots) or 4 ((k >> 1) & 1)
  //      (8 slots): a transposing read takes 64 bytes from each of four consecutive keys, which the swizzle (with 12
  //      slots the pitch itself) spreads over the four quarters of the banks.
  // With 8 and 16 slots both swizzles depend on the row only through bits the lane's position fixes, so each lane keeps
  // one byte offset per operand and advances it by a tile per load; 12 slots do not divide the 256 lanes, and each load
  // of a tile has an offset of its own.  Lanes whose chunk lies past the head size sit at an offset that stays out of range.
  const uint32_t k_bytes = kl > 0 ? (uint32_t)(((int64_t)(kl - 1) * a.k_ss + a.D) * E::kSize) : 0u;
  const uint32_t v_bytes = kl > 0 ? (uint32_t)(((int64_t)(kl - 1) * fa.v_ss + a.D) * E::kSize) : 0u;
  const desc_t k_desc = make_desc(kbase, k_bytes);
  const desc_t v_desc = make_desc(vbase, v_bytes);
  const uint32_t k_row_bytes = (uint32_t)(a.k_ss * E::kSize), v_row_bytes = (uint32_t)(fa.v_ss * E::kSize);
  constexpr int NOFF = DP == 96 ? KLOADS : 1;
  uint32_t k_off[NOFF], v_off[NOFF];
#pragma unroll
  for (int i = 0; i < NOFF; ++i) {
    const int row = (i * kBlock + tid) / KVEC_ROW, slot = (i * kBlock + tid) % KVEC_ROW;
    const int k_c = slot ^ kswz(row), v_c = slot ^ vswz(row);
    k_off[i] = (k_c * EPV < a.D) ? row * k_row_bytes + k_c * EPV * E::kSize : kOutOfRange;
    v_off[i] = (v_c * EPV < a.D) ? row * v_row_bytes + v_c * EPV * E::kSize : kOutOfRange;
  }
  auto fetch_tile = [&](const desc_t &desc, T *dst, uint32_t (&off)[NOFF], uint32_t row_bytes) {
    const uint32_t lds = lds_address(dst) + wave * kWave * 16;
#pragma unroll
    for (int i = 0; i < KLOADS; ++i)
      buffer_load16_to_lds(desc, lds + i * kBlock * 16, NOFF > 1 ? off[i % NOFF] : off[0] + i * (kBlock / KVEC_ROW) * row_bytes);
#pragma unroll
    for (int i = 0; i < NOFF; ++i) off[i] += BK * row_bytes;
  };
  auto fetch_k = [&](T *dst) { fetch_tile(k_desc, dst, k_off, k_row_bytes); };
  auto fetch_v = [&](T *dst) { fetch_tile(v_desc, dst, v_off, v_row_bytes); };
  // fragment addresses.  K: row 32 kb + r, chunk 2 vs + g.  V (transposing read): lane j of a 16-lane group
  // points at key j / 4 of the group's four keys and at channels 4 (j % 4) .. + 3 of the group's sixteen; the
  // read hands lane i of the group channel i of those sixteen at the four keys.
  const int ksw = kswz(r);
  const int tj = lane & 15, tg = (lane >> 4) & 1;     // position in the 16-lane group; which half of a 32-channel tile
  const int vsw = vswz(tj >> 2) / 4;
  uint32_t v_frag[DMT];                                // byte offset of this lane's read for channel tile mt, keys 4g + 0..3
#pragma unroll
  for (int mt = 0; mt < DMT; ++mt)
    v_frag[mt] = (uint32_t)((4 * g + (tj >> 2)) * ROW * E::kSize + (4 * (mt ^ vsw) + 2 * tg + ((tj >> 1) & 1)) * 16 + (tj & 1) * 8);

  floatx16 o[DMT];
#pragma unroll
  for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
    for (int x = 0; x < 16; ++x) o[mt][x] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const float c_exp = fa.scale * kLog2e;
  // The running maximum is only moved (and the accumulators rescaled) when some query's new
  // maximum exceeds it by more than 2^8 after scaling: until then probabilities are formed
  // against the older, slightly smaller maximum and stay below 2^8, well inside the 16-bit
  // range, and the final division by the row sum cancels the common factor.
  const float lazy_gap = 8.0f / c_exp;

  // K tile kt is read out of buffer kt & 1 while K tile kt + 1 travels into the other one.  Two V buffers: V goes the
  // same way, one barrier per tile.  One V buffer: V tile kt is sent for at the top of iteration kt (its buffer was in use
  // until the barrier that ended iteration kt - 1) and waited for between the softmax and the second contraction, two
  // barriers per tile.
  fetch_k(lds_k[0]);
  if constexpr (NVB == 2) fetch_v(lds_v[0]);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NVB == 2 ? 2 : 1) * KLOADS) : "memory");
  // the wave's own Q rows have landed; the barrier below keeps the tiles of the key loop off them until all have read
#pragma unroll
  for (int vs = 0; vs < NVS; ++vs)
    qf[vs] = *reinterpret_cast<const uint4 *>(&q_stage[r * ROW + (((2 * vs + g) ^ ksw) * EPV)]);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NVB == 2 ? KLOADS : 0) : "memory");
  lds_barrier();

  for (int kt = 0; kt < nkt; ++kt) {
    const int k0 = kt * BK;
    const T *ksrc = lds_k[kt & 1];
    const T *vsrc = lds_v[NVB == 2 ? kt & 1 : 0];
    if constexpr (NVB == 2) {
      fetch_k(lds_k[(kt + 1) & 1]);              // tiles kt + 1 (past the end: out of range, zeros, no traffic)
      fetch_v(lds_v[(kt + 1) & 1]);
    } else {
      fetch_v(lds_v[0]);                         // V tile kt
      fetch_k(lds_k[(kt + 1) & 1]);              // K tile kt + 1
    }
    uint4 pf[KB * 2];                            // B operands of the second MFMA: the probabilities of this tile
    const bool live = k0 < vis_max;              // wave-uniform: later tiles are masked for all of this wave's queries

    if (live) {
      // ---- S^T = K Q^T; the K fragments are read from LDS a step ahead of the MFMAs
      floatx16 s[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int x = 0; x < 16; ++x) s[kb][x] = 0.f;
      {
        uint4 kf[2][KB];                             // fragments of the step after the one the MFMAs work on
        auto load_step = [&](int vs, uint4 (&dst)[KB]) {
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
            dst[kb] = *reinterpret_cast<const uint4 *>(&ksrc[(kb * 32 + r) * ROW + (((2 * vs + g) ^ ksw) * EPV)]);
        };
        load_step(0, kf[0]);
#pragma unroll
        for (int vs = 0; vs < NVS; ++vs) {
          if (vs + 1 < NVS) load_step(vs + 1, kf[(vs + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);         // keep the reads of the next step ahead of these MFMAs
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) M::step(kf[vs & 1][kb], qf[vs], s[kb]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }

      // ---- mask + online softmax; register 4j+i of block kb holds key k0 + 32kb + 8j + 4g + i
      float m_tile = -INFINITY;
      if (k0 + BK <= vis_min) {  // whole tile visible to every query of this wave: no masking work
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int x = 0; x < 16; ++x) m_tile = fmaxf(m_tile, s[kb][x]);
      } else {
        // this lane's query and the keys it may see (k < vis_l), counted afresh: only the tiles on the diagonal come here
        const int l = lane_now(), ql_ = q0 + wave * 32 + (l & 31);
        const int vis_l = ((unsigned)ql_ < (unsigned)ql) ? (a.causal ? min(kl, ql_ + (kl - ql) + 1) : kl) : 0;
        const int lim = vis_l - k0 - 4 * (l >> 5);   // register (kb, x) is visible iff 32kb + 8(x/4) + x%4 < lim
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int x = 0; x < 16; ++x) {
            const float v = (kb * 32 + 8 * (x >> 2) + (x & 3) < lim) ? s[kb][x] : -INFINITY;
            s[kb][x] = v;
            m_tile = fmaxf(m_tile, v);
          }
      }
      {  // the other half of this query's keys sits in lane r + 32
        float lo, hi;
        halves_of(m_tile, lo, hi);
        m_tile = fmaxf(lo, hi);
      }
      if (__builtin_amdgcn_ballot_w64(m_tile - lazy_gap > m_run) != 0) {   // -inf + gap stays -inf: the first tile moves it
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
      for (int kb = 0; kb < KB; ++kb) {
        Pack<T, EPV> pk[2];
#pragma unroll
        for (int x = 0; x < 16; ++x) {
          // exp2(-inf) is 0, so masked keys need no special case
          const float p = __builtin_amdgcn_exp2f(fmaf(s[kb][x], c_exp, moff));
          l_tile += p;
          pk[x >> 3].v[x & 7] = E::from_float(p);                // group t = x/8 takes registers j = 2t, 2t+1
        }
        pf[2 * kb] = __builtin_bit_cast(uint4, pk[0]);
        pf[2 * kb + 1] = __builtin_bit_cast(uint4, pk[1]);
      }
      l_run += l_tile;

    }

    // One V buffer: V tile kt was sent for before K tile kt + 1 and the loads complete in order: it has landed once only
    // the K loads are outstanding; the barrier publishes every wave's share
    if constexpr (NVB == 1) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(KLOADS) : "memory");
      lds_barrier();
    } else if (kt == 0) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * KLOADS) : "memory");
      lds_barrier();
    }

    if (live) {
      // ---- O^T += V^T P^T; the A operand reads V at the keys the B registers hold:
      //      elements 0..3 <-> keys 16gi + 4g + 0..3, elements 4..7 <-> keys 16gi + 8 + 4g + 0..3
      constexpr int NG = KB * 2;                      // groups of 16 keys
      uint4 va[2][DMT];
      auto load_group = [&](int gi, uint4 (&dst)[DMT]) {
        const char *vt = reinterpret_cast<const char *>(vsrc) + gi * 16 * ROW * E::kSize;
#pragma unroll
        for (int mt = 0; mt < DMT; ++mt) {
          const uint2 lo = lds_read_tr16(vt + v_frag[mt]);                          // keys 16 gi + 4 g + 0..3
          const uint2 hi = lds_read_tr16(vt + v_frag[mt] + 8 * ROW * E::kSize);     // keys 16 gi + 8 + 4 g + 0..3
          dst[mt] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
      };
      load_group(0, va[0]);
#pragma unroll
      for (int gi = 0; gi < NG; ++gi) {
        if (gi + 1 < NG) load_group(gi + 1, va[(gi + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mt = 0; mt < DMT; ++mt) M::step(va[gi & 1][mt], pf[gi], o[mt]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }

    // The next tiles have landed once none of this wave's loads is outstanding; the barrier publishes them and
    // frees the buffers of this one
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
  }

  // ---- normalise and store: register 4j+i of tile mt holds channel 32mt + 8j + 4g + i of this lane's query
  // each half of the wave has added up its own keys: both were scaled alike, so they are put together once
  float l_lo, l_hi;
  halves_of(l_run, l_lo, l_hi);
  const float l_all = l_lo + l_hi, inv = l_all > 0.f ? 1.0f / l_all : 0.f;
  const int lane_e = lane_now(), r_e = lane_e & 31, g_e = lane_e >> 5;
  if (NORM || fa.c_vec16) {
    // A lane holds 8-byte pieces of its own row, 32 rows per store instruction; through LDS (the K buffers are free
    // behind the loop's last barrier, each wave takes the 32 rows' worth that is its own, so no barrier is needed)
    // the wave's tile leaves as whole rows: 16 bytes per lane, four to eight rows per instruction.  Chunk c of row r
    // sits in slot c ^ oswz(r): writes and reads both spread over all banks.
    auto oswz = [](int row) { return DP == 96 ? (row >> 2) & 3 : row & (KVEC_ROW - 1); };
    const rsrc_t c_rsrc = make_rsrc(cbase, (uint32_t)(((int64_t)(ql - 1) * fa.c_ss + a.D) * E::kSize));
    char *stage = reinterpret_cast<char *>(&lds_k[0][0]) + wave * 32 * ROW * E::kSize;
#pragma unroll
    for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        Pack<T, 4> pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk.v[i] = E::from_float(o[mt][4 * j + i] * inv);
        const int c = 4 * mt + j;
        *reinterpret_cast<Pack<T, 4> *>(stage + r_e * ROW * E::kSize + ((c ^ oswz(r_e)) * 16) + g_e * 8) = pk;
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's own writes, before its lanes read each other's
#pragma unroll
    for (int i = 0; i < 32 * KVEC_ROW / kWave; ++i) {
      const int row = (i * kWave + lane_e) / KVEC_ROW, c = (i * kWave + lane_e) % KVEC_ROW;
      const uint4 v = *reinterpret_cast<const uint4 *>(stage + row * ROW * E::kSize + ((c ^ oswz(row)) * 16));
      const int qrow = q0 + wave * 32 + row;
      if constexpr (NORM) {
        const uint32_t at = (uint32_t)((int64_t)qrow * fa.c_ss + c * EPV) * E::kSize;
        buffer_store16<kAgentScope>(c_rsrc, (unsigned)qrow < (unsigned)ql && c * EPV < a.D ? at : kOutOfRange, v);
        continue;
      }
      if ((unsigned)qrow < (unsigned)ql && c * EPV < a.D) *reinterpret_cast<uint4 *>(cbase + (int64_t)qrow * fa.c_ss + c * EPV) = v;
    }
    if constexpr (NORM) {
      norm_tile<DT, DP>(*norm, rows);
    }
    return;
  }
  const int q_e = q0 + wave * 32 + r_e;
  if ((unsigned)q_e >= (unsigned)ql) return;
  T *crow = cbase + (int64_t)q_e * fa.c_ss;
#pragma unroll
  for (int mt = 0; mt < DMT; ++mt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = mt * 32 + 8 * j + 4 * g_e;
      if (d < a.D) {
        Pack<T, 4> pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk.v[i] = E::from_float(o[mt][4 * j + i] * inv);
        store_pack<T, 4>(crow + d, pk);
      }
    }
}

template <int DT, int DP, int NVS, bool Q_ONCE>
__global__ __launch_bounds__(kBlock, DP == 64 ? 4 : 3) void attn_fused_kernel(FusedArgs fa) {
  fused_tile<DT, DP, NVS, false, Q_ONCE>(fa, nullptr);
}
template <int DT, int DP, int NVS>
__global__ __launch_bounds__(kBlock, DP == 64 ? 4 : 3) void attn_fused_norm_kernel(FusedArgs fa, NormArgs norm) {
  fused_tile<DT, DP, NVS, true, false>(fa, &norm);
}

// The attention and, in workgroups of their own, a residual + LayerNorm that does not read its output (a row-parallel
// projection lies between them).  The attention is bound by instruction issue and by the chain of its longest workgroup, the
// rows by memory: side by side they take less than one after the other, and a launch less.  us a layer, two launches / one:
// 14213 tokens, 12 heads x 128, rows of 12288 252 / 240; 3485, 32 x 128, 8192 114 / 107; 3569, 16 x 64, 8192 49 / 43.5;
// 3866, 10 x 80, 3200 42 / 32; 1033, 8 x 64, 2048 19.3 / 15.7; 300, 5 x 64, 640 18.3 / 15.3.  (Rows of 14336, which a
// workgroup could hold with one load in flight less: 170 / 182, so 12288 is where it ends.)
template <int DT, int DP, int NVS, bool Q_ONCE, bool STREAM>
__global__ __launch_bounds__(kBlock, DP == 64 ? 4 : 3) void attn_fused_beside_norm_kernel(FusedArgs fa, NormRows rows) {
  const int j = blockIdx.x / kXcds, x = blockIdx.x % kXcds;
  const int before = min((int)(((uint64_t)j * rows.step) >> 16), rows.groups);
  const int behind = min((int)(((uint64_t)(j + 1) * rows.step) >> 16), rows.groups);
  if (behind > before) norm_rows<DT, STREAM>(rows, before * kXcds + x);
  else fused_tile<DT, DP, NVS, false, Q_ONCE>(fa, nullptr, (j - before) * kXcds + x);
}

template <int DT, int DP, int NVS, bool Q_ONCE = false>
static void launch_form(const FusedArgs &fa, const NormArgs *norm, const NormRows *rows, unsigned grid, hipStream_t s) {
  if (rows) {
    grid += (unsigned)rows->groups * kXcds;
    constexpr bool ONCE = Q_ONCE && DP == 128;
    if (rows->rows * rows->width * 2 >= kStreamStoreBytes) attn_fused_beside_norm_kernel<DT, DP, NVS, ONCE, true><<<grid, kBlock, 0, s>>>(fa, *rows);
    else attn_fused_beside_norm_kernel<DT, DP, NVS, ONCE, false><<<grid, kBlock, 0, s>>>(fa, *rows);
  } else if (norm) attn_fused_norm_kernel<DT, DP, NVS><<<grid, kBlock, 0, s>>>(fa, *norm);
  else attn_fused_kernel<DT, DP, NVS, Q_ONCE><<<grid, kBlock, 0, s>>>(fa);
}

// Q is read once, and non-temporal it leaves the caches to what is read again, K and V by the unit's other tiles and the context by the
// LayerNorm.  That pays with heads of 128 channels, whose Q rows are whole 128-byte lines, and hardly with 96 (a line and a half); the
// others lose, their lines being shared with the rows beside them.  us, cached / non-temporal:
//   128: 4 layers of 8 sequences of up to 512, 32 heads 154.4 / 150.5, 6 of 16 of up to 256, 32 241 / 236, 6 of 64 of up to 40, 20 143.4 /
//     141.7, 4 of 3 of up to 700, 72, no mask 245.6 / 242.5, 4 of 16 of up to 1024, 56 864 / 858; with the LayerNorm's rows beside it 6 of 40
//     of up to 128, 24 365 / 357, 8 of 1 of up to 100, 12 97.5 / 97.5, 4 of 16 of up to 512, 32 327 / 326;
//   96: 6 of 8 of up to 200, 32 121 / 119, 4 of 4 of up to 1000, 24 213 / 211, 6 of 24 of up to 256, 20 173.8 / 174.4; rows beside it 6 of 24 of
//     up to 256, 20 243.5 / 250.3, 6 of 8 of up to 600, 16 235.6 / 241.4;
//   others: 80 channels 4 of 7 of up to 1531, 20 231 / 235, 6 of 16 of up to 400, 20, rows beside it 297 / 306; 112 6 of 16 of up to 512, 24
//     290 / 297; 120 6 of 40 of up to 100, 40 277 / 283; 64 12 of 39 of up to 557, 5 304 / 316.
// With the LayerNorm in the launch K and V of all tiles come in at once, and it loses at 128 too: 4 of 4 of up to 700, 16 114 / 116.
template <int DT>
static int launch_fused(FusedArgs &fa, const NormArgs *norm, const NormRows *rows, hipStream_t s) {
  const AttnArgs &a = fa.base;
  const unsigned grid = (unsigned)(ceil_div(a.units, kXcds) * kXcds * a.ntq);
  if (a.D <= 64) launch_form<DT, 64, 4>(fa, norm, rows, grid, s);
  else if (a.D <= 80) launch_form<DT, 96, 5>(fa, norm, rows, grid, s);
  else if (a.D < 96) launch_form<DT, 96, 6>(fa, norm, rows, grid, s);
  else if (a.D == 96) launch_form<DT, 96, 6, true>(fa, norm, rows, grid, s);
  else if (a.D < 128) launch_form<DT, 128, 8>(fa, norm, rows, grid, s);
  else launch_form<DT, 128, 8, true>(fa, norm, rows, grid, s);
  EN_RETURN_IF_LAUNCH_FAILED();
  return EN_OK;
}

}  // namespace en

extern "C" int en_attn_fused_query_tile(int q_seq_len, int k_seq_len, int size_per_head, int causal, int dtype) {
  // The 256-row tile (64 queries per wave, fused_wide.hip) halves the LDS reads, tile loads and barriers per FLOP
  // but runs two waves per SIMD instead of three, and measures slower on every shape tried (uniform 1024-key
  // rows, 64 heads: 778 against 906 TFLOP/s; ragged batches lose more, having fewer and longer workgroups):
  // never chosen by itself.
  (void)q_seq_len; (void)k_seq_len; (void)size_per_head; (void)causal;
  return dtype == EN_F32 ? 64 : en::kQTile;     // fp32: the kernel of fused_f32.hip, 64-row tiles
}

namespace en {

static int attn_fused(const void *q, const void *k, const void *v, void *ctx, const int32_t *k_lens, const
                      int32_t *q_lens, int batch, int head_num, int q_seq_len, int k_seq_len, int size_per_head, const int64_t
                      *q_strides, const int64_t *k_strides, const int64_t *v_strides, const int64_t *c_strides, const int32_t
                      *q_row_offsets, const int32_t *k_row_offsets, float scale, int causal, int dtype, const int32_t
                      *tile_table, int query_tile, const NormArgs *norm, const NormRows *rows, en_stream_t stream) {
  if (!q || !k || !v || !ctx || !k_lens || !q_strides || !k_strides || !v_strides || !c_strides) return EN_ERR_NULL;
  if (batch < 1 || head_num < 1 || q_seq_len < 1 || k_seq_len < 1 || size_per_head < 1) return EN_ERR_SHAPE;
  if (dtype != EN_F16 && dtype != EN_BF16 && dtype != EN_F32) return EN_ERR_DTYPE;
  const bool f32 = dtype == EN_F32;
  const int es = f32 ? 4 : 2, epv = 16 / es;
  if (size_per_head > 128 || (size_per_head % epv) != 0) return EN_ERR_UNSUPPORTED;
  if (f32 && size_per_head > 64) return EN_ERR_UNSUPPORTED;   // the fp32 kernel is built for heads of up to 64 channels
  if (!(scale > 0.f)) return EN_ERR_UNSUPPORTED;  // masked scores are -inf; -inf * 0 would not stay masked
  if (query_tile == 0) query_tile = en_attn_fused_query_tile(q_seq_len, k_seq_len, size_per_head, causal, dtype);
  if (f32 ? query_tile != 64 : (query_tile != kQTile && query_tile != kWideQTile)) return EN_ERR_UNSUPPORTED;
  if (query_tile == kWideQTile && size_per_head <= 64) return EN_ERR_UNSUPPORTED;   // the 64-query wave is built for 65..128 channels
  if ((int64_t)batch * head_num > INT32_MAX / 64) return EN_ERR_SHAPE;
  if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(v, 16) || !aligned_to(ctx, 4 * es)) return EN_ERR_ALIGN;
  for (int i = 0; i < 3; ++i) {
    if ((q_strides[i] % epv) || (k_strides[i] % epv) || (v_strides[i] % epv) || (c_strides[i] % 4)) return EN_ERR_ALIGN;
    if (q_strides[i] < 0 || k_strides[i] < 0 || v_strides[i] < 0 || c_strides[i] < 0) return EN_ERR_UNSUPPORTED;
  }
  // 32-bit byte offsets, advanced a tile at a time up to two tiles past the end
  if ((int64_t)q_seq_len * q_strides[2] * es >= (1ll << 31) || ((int64_t)k_seq_len + 256) * k_strides[2] * es >= (1ll << 31) ||
      ((int64_t)k_seq_len + 256) * v_strides[2] * es >= (1ll << 31))
    return EN_ERR_UNSUPPORTED;
  if (f32 && tile_table) return EN_ERR_UNSUPPORTED;            // the table lists 128- or 256-row tiles; the fp32 kernel has 64-row ones
  FusedArgs fa{};
  AttnArgs &a = fa.base;
  a.a_ptr = q; a.b_ptr = k; a.out = ctx; a.k_lens = k_lens; a.q_lens = q_lens;
  a.B = batch; a.H = head_num; a.Sq = q_seq_len; a.Sk = k_seq_len; a.D = size_per_head;
  a.q_sb = q_strides[0]; a.q_sh = q_strides[1]; a.q_ss = q_strides[2];
  a.k_sb = k_strides[0]; a.k_sh = k_strides[1]; a.k_ss = k_strides[2];
  a.alpha = 1.f; a.causal = causal ? 1 : 0;
  a.ntq = (int)ceil_div(q_seq_len, kQTile);
  a.units = batch * head_num;
  fa.v = v;
  fa.v_sb = v_strides[0]; fa.v_sh = v_strides[1]; fa.v_ss = v_strides[2];
  fa.c_sb = c_strides[0]; fa.c_sh = c_strides[1]; fa.c_ss = c_strides[2];
  fa.q_row0 = q_row_offsets; fa.k_row0 = k_row_offsets;
  fa.c_vec16 = aligned_to(ctx, 16) && (c_strides[0] % epv) == 0 && (c_strides[1] % epv) == 0 && (c_strides[2] % epv) == 0;
  if (tile_table && q_lens) return EN_ERR_UNSUPPORTED;      // the table lists the query tiles of min(k_lens, q_seq_len) rows
  a.tile_table = tile_table;
  fa.scale = scale;
  hipStream_t s = (hipStream_t)stream;
  if (norm && (!fa.c_vec16 || query_tile == kWideQTile)) return EN_ERR_UNSUPPORTED;
  if (rows && (f32 || query_tile == kWideQTile)) return EN_ERR_UNSUPPORTED;
  if (f32) return launch_fused_f32(fa, norm, s);
  if (query_tile == kWideQTile) {
    a.ntq = (int)ceil_div(q_seq_len, kWideQTile);
    return launch_fused_wide(dtype, fa, s);
  }
  return dtype == EN_F16 ? launch_fused<EN_F16>(fa, norm, rows, s) : launch_fused<EN_BF16>(fa, norm, rows, s);
}

// Workgroups that are resident at once: what LDS and registers leave room for on 256 CUs.
static int64_t resident_workgroups(int size_per_head, int dtype) { return dtype == EN_F32 ? 512 : size_per_head <= 64 ? 1024 : 768; }

// Where one launch is the faster form, us per layer, one launch / two (6 layers, hot operands, launches queued ahead of the GPU).  Meeting costs about 6 us
// (context written through, counted, seen, read back), a trip to memory for every round of a wave's rows (norm_rows_ahead); a
// LayerNorm launch costs 5 us and what its bytes take.
//   16-bit: context of 7 MB and more and at most three rows per wave: 24 sequences of up to 384, 16 heads x 64 19.1 / 21.1, 32 of up
//     to 512, 12 x 64 20.9 / 23.1, 8 of up to 665, 14 x 96 22.0 / 22.8.  That is where the two met while two rows of a wave were in
//     flight; now that three go out at once they meet near 3 MB (8 of up to 300, 12 x 80 13.8 / 13.1; 32 of up to 128, 16 x 64, 4.0 MB
//     12.25 / 12.2), and the line leaves up to 1 us a layer from there to 7 MB (8 of up to 256, 32 x 64 13.3 / 13.6, 24 of up to 300,
//     12 x 64 14.5 / 15.0, 14 of up to 356, 11 x 80 17.0 / 18.0, 4 of up to 700, 16 x 128 22.8 / 23.7, 1 of 1024 29.4 / 29.6).  Smaller
//     ones lose (16 of up to 128, 12 x 64 10.7 / 9.5, one of 509 15.1 / 13.4), as do few heads (64 of up to 128, 4 x 64 15.1 / 10.5).
//     Short prompts: where the host is what bounds a layer, one launch less is what counts (one of 60 rows, 12 x 64 10.4 / 11.3, 64 of
//     up to 30, 4 x 64 10.7 / 13.1).  The GPU alone takes longer for it: 8.2 / 7.35 and 8.4 / 7.3, 64 of up to 64, 8 x 64 9.35 / 8.8,
//     32 of up to 64, 16 x 64 9.3 / 9.15.
//   fp32 (64-row tiles): 4 of up to 128, 12 x 64 15.0 / 15.5, 21 of up to 73, 6 x 64 12.3 / 12.5; 58 of up to 239, 3 x 64 39.0 / 34.8.
static bool one_launch_pays(int heads, int seq_len, int64_t tiles, int64_t bytes, int dtype) {
  const int64_t per_wave = ceil_div(std::min(seq_len, dtype == EN_F32 ? kF32QTile : kQTile), heads * (kBlock / kWave));
  if (dtype == EN_F32) return per_wave <= 2;
  return (bytes >= 7 << 20 && per_wave <= 3) || (seq_len <= 64 && per_wave <= 2 && tiles * heads <= 512);
}

// Query tiles of a batch: half a tile a sequence is the ragged one, on average.
static int64_t query_tiles(int batch, int max_seq_len, int64_t total_tokens, int dtype) {
  const int64_t tile = dtype == EN_F32 ? kF32QTile : kQTile;
  return max_seq_len <= tile ? batch : total_tokens / tile + (batch + 1) / 2;
}

constexpr int kNormPolls = 64;      // looks at a meeting word before a workgroup leaves its rows to the last one: tens of us

static bool overlap(const void *a, int64_t a_bytes, const void *b, int64_t b_bytes) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return x < y + (uintptr_t)b_bytes && y < x + (uintptr_t)a_bytes;
}

int attn_fused_beside_norm(const void *qkv, void *ctx, const int32_t *seq_lens, const int32_t *cu_seqlens, int batch, int head_num,
                           int max_seq_len, int size_per_head, int64_t total_tokens, float scale, int causal, int dtype,
                           const int32_t *tile_table, const void *in, const void *residual, int64_t residual_rows,
                           const int32_t *residual_row_offsets, const void *gamma, const void *beta, void *y, int64_t hidden,
                           float eps, en_stream_t stream) {
  if (dtype != EN_F16 && dtype != EN_BF16) return EN_ERR_UNSUPPORTED;
  if (batch < 1 || head_num < 1 || max_seq_len < 1 || size_per_head < 1 || total_tokens < 1) return EN_ERR_SHAPE;
  const int64_t T = total_tokens, D = size_per_head, width = head_num * D, out_bytes = T * hidden * 2, ctx_bytes = T * width * 2;
  if (hidden % 8 || hidden / 8 > kNormRowsMaxVectors || T > INT32_MAX) return EN_ERR_UNSUPPORTED;
  for (const void *p : {in, residual, gamma, beta, (const void *)y})
    if (!aligned_to(p, 16)) return EN_ERR_UNSUPPORTED;
  // Each role reads while the other writes: buffers that a caller has laid over each other need two launches.
  const int64_t meta = ((int64_t)batch + 1) * 4;
  if (overlap(ctx, ctx_bytes, in, out_bytes) || overlap(ctx, ctx_bytes, residual, residual_rows * hidden * 2) ||
      overlap(ctx, ctx_bytes, gamma, hidden * 2) || overlap(ctx, ctx_bytes, beta, hidden * 2) ||
      (residual_row_offsets && overlap(ctx, ctx_bytes, residual_row_offsets, T * 4)) || overlap(y, out_bytes, ctx, ctx_bytes) ||
      overlap(y, out_bytes, qkv, 3 * ctx_bytes) || overlap(y, out_bytes, seq_lens, meta - 4) || overlap(y, out_bytes, cu_seqlens, meta) ||
      (tile_table && overlap(y, out_bytes, tile_table, en_attn_tile_table_elems(batch, head_num, max_seq_len, 0) * 4)))
    return EN_ERR_UNSUPPORTED;
  NormRows rows{in, residual, residual_row_offsets, gamma, beta, y, T, (int)hidden, eps, 0, 0};
  rows.groups = (int)ceil_div(ceil_div(T, norm_rows_per_workgroup((int)hidden)), kXcds);
  // Rows are dealt out between the attention's workgroups, as if those were twice their likely number: the long ones, which
  // come first, start the earlier for it (10 heads x 80, 3866 tokens: 34 us by the likely number itself, 32 by twice that); but
  // over no more groups than the launch has for the attention: all groups of rows then come before its last one, and no
  // workgroup looks behind the end of the tile table.
  const int64_t attention = std::min(2 * ceil_div(query_tiles(batch, max_seq_len, T, dtype) * head_num, kXcds),
                                     ceil_div((int64_t)batch * head_num, kXcds) * ceil_div(max_seq_len, kQTile));
  rows.step = (uint32_t)ceil_div((int64_t)rows.groups << 16, attention + rows.groups);
  const char *pk = static_cast<const char *>(qkv);
  const int64_t in_strides[3] = {0, 3 * D, 3 * width}, out_strides[3] = {0, D, width};
  return attn_fused(pk, pk + D * 2, pk + 2 * D * 2, ctx, seq_lens, nullptr, batch, head_num, max_seq_len, max_seq_len, size_per_head,
                    in_strides, in_strides, in_strides, out_strides, cu_seqlens, cu_seqlens, scale, causal, dtype, tile_table, 0,
                    nullptr, &rows, stream);
}

}  // namespace en

extern "C" {

int64_t en_attn_fused_norm_arrivals(int batch, int q_seq_len) {
  return batch < 1 || q_seq_len < 1 ? 0 : batch * en::ceil_div(q_seq_len, en::kF32QTile) * en::kNormWordStride;      // the lower of the tile heights
}

int en_attn_fused_norm_pays(int batch, int head_num, int max_seq_len, int size_per_head, int64_t total_tokens, int dtype) {
  const int es = en::dtype_size(dtype);
  if (!es || batch < 1 || head_num < 1 || max_seq_len < 1 || size_per_head < 1 || total_tokens < 1) return 0;
  return en::one_launch_pays(head_num, max_seq_len, en::query_tiles(batch, max_seq_len, total_tokens, dtype),
                             total_tokens * head_num * size_per_head * es, dtype);
}

int en_attn_fused_norm(const void *qkv, void *ctx, const int32_t *seq_lens, const int32_t *cu_seqlens, int batch, int head_num,
                       int max_seq_len, int size_per_head, int64_t total_tokens, float scale, int causal, int dtype,
                       const int32_t *tile_table, const void *hidden_padded, const int32_t *residual_row_offsets, const void *gamma,
                       const void *beta, void *y, float eps, uint64_t *arrivals, int polls, en_stream_t stream) {
  using namespace en;
  if (!qkv || !ctx || !seq_lens || !cu_seqlens || !hidden_padded || !residual_row_offsets || !gamma || !beta || !y || !arrivals)
    return EN_ERR_NULL;
  const int es = dtype_size(dtype);
  if (!es) return EN_ERR_DTYPE;
  if (batch < 1 || head_num < 1 || max_seq_len < 1 || size_per_head < 1 || total_tokens < 1) return EN_ERR_SHAPE;
  const int64_t width = (int64_t)head_num * size_per_head, T = total_tokens;
  if (head_num > kNormMaxHeads || width * es % 16 || width * es / 16 > kNormMaxVectors) return EN_ERR_UNSUPPORTED;
  if ((int64_t)max_seq_len * width * es >= (1ll << 31)) return EN_ERR_UNSUPPORTED;              // 32-bit offsets into a sequence's context
  for (const void *p : {qkv, (const void *)ctx, hidden_padded, gamma, beta, (const void *)y})
    if (!aligned_to(p, 16)) return EN_ERR_UNSUPPORTED;
  // Workgroups that wait for one another hold their place, so all of them have to be resident at once.
  if (query_tiles(batch, max_seq_len, T, dtype) * head_num > resident_workgroups(size_per_head, dtype)) return EN_ERR_UNSUPPORTED;
  if (polls < 0 && !en_attn_fused_norm_pays(batch, head_num, max_seq_len, size_per_head, T, dtype)) return EN_ERR_UNSUPPORTED;
  // Rows are normalised while other tiles still read: buffers that a caller has laid over each other need two launches.
  const int64_t bytes = T * width * es, meta = ((int64_t)batch + 1) * 4;
  for (const void *p : {(const void *)ctx, (const void *)y}) {
    if (overlap(p, bytes, qkv, 3 * bytes) || overlap(p, bytes, seq_lens, meta - 4) || overlap(p, bytes, cu_seqlens, meta) ||
        overlap(p, bytes, gamma, width * es) || overlap(p, bytes, beta, width * es) || overlap(p, bytes, residual_row_offsets, T * 4) ||
        overlap(p, bytes, hidden_padded, (int64_t)batch * max_seq_len * width * es))
      return EN_ERR_UNSUPPORTED;
  }
  if (overlap(ctx, bytes, y, bytes)) return EN_ERR_UNSUPPORTED;
  // A captured launch may run again on any stream, beside launches that use the same meeting words.
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &capture) != hipSuccess) {      // e.g. the null stream beside a capture
    (void)hipGetLastError();
    return EN_ERR_UNSUPPORTED;
  }
  if (capture != hipStreamCaptureStatusNone) return EN_ERR_UNSUPPORTED;
  const NormArgs norm{hidden_padded, residual_row_offsets, gamma, beta, ctx, y, reinterpret_cast<unsigned long long *>(arrivals),
                      (int)width, polls < 0 ? kNormPolls : polls, eps};
  const char *pk = static_cast<const char *>(qkv);
  const int64_t D = size_per_head, in_strides[3] = {0, 3 * D, 3 * width}, out_strides[3] = {0, D, width};
  return attn_fused(pk, pk + D * es, pk + 2 * D * es, ctx, seq_lens, nullptr, batch, head_num, max_seq_len, max_seq_len, size_per_head,
                    in_strides, in_strides, in_strides, out_strides, cu_seqlens, cu_seqlens, scale, causal, dtype,
                    dtype == EN_F32 ? nullptr : tile_table, 0, &norm, nullptr, stream);
}

int en_attn_fused(const void *q, const void *k, const void *v, void *ctx, const int32_t *k_lens,
                             const int32_t *q_lens, int batch, int head_num, int q_seq_len, int k_seq_len,
                             int size_per_head, const int64_t *q_strides, const int64_t *k_strides,
                             const int64_t *v_strides, const int64_t *c_strides, const int32_t *q_row_offsets,
                             const int32_t *k_row_offsets, float scale, int causal, int dtype,
                             const int32_t *tile_table, int query_tile, en_stream_t stream) {
  return en::attn_fused(q, k, v, ctx, k_lens, q_lens, batch, head_num, q_seq_len, k_seq_len,
                        size_per_head, q_strides, k_strides, v_strides, c_strides, q_row_offsets, k_row_offsets, scale, causal,
                        dtype, tile_table, query_tile, nullptr, nullptr, stream);
}

}  // extern "C"
