// fbs_layers.hip - teacher-forced positions layer by layer: prompts taken in before a choice, and
// rows whose every position is scored.
//
// The step (RS stack/session.rs:4129-4403) runs one position after another because the next token
// is not known before the writer chose it. Where every token is known, only the recurrence's
// transport ties a position to the one before: a layer's norms, gathers, rotations, gates,
// requantizes and feed-forward block depend on the layer's input at that position alone, and the
// causal window on the drives of earlier positions. So these calls run each layer over all positions
// at once, in two kernels a layer: fbs_layer_front (a wavefront a position: the end of the layer
// before and the start of this one, up to the drives, the transitions and the output gates) and
// fbs_layer_chain (a lane a channel of a sequence: windows and transport). A chain step is some 50
// instructions against the step's 2,000 a layer, so a prompt's time is set by the positions' work spread
// over the chip and no longer by the step's serial chain. The choices come from fbs_layer_query (final
// norm, Q12 query and drawer selection of each position), fbs_layer_lists and a drawer-major scan that
// reads a member row once for the queries that kept its drawer.
// Every value is formed by the step's own routines (fbs_run.h), so the results are its bit for bit.
// At width 256 (6 layers, window 16), 300 prompts of 509 tokens: 19.2 ms by steps, 3.8 by layers (front
// 448 us a layer, chain 214); 8,192 rows of 128 76 and 40 ms.
#include "fbs_layers.h"

#include <type_traits>

#include "fbs_run.h"

namespace fbs {

namespace {

constexpr uint32_t kFrontWaves = 4;  // wavefronts a block of fbs_layer_front, a position each
constexpr uint32_t kChainWaves = 2;  // wavefronts a block of fbs_layer_chain: the transport and the windows
constexpr uint32_t kRound = 8;       // positions of a round
constexpr uint32_t kStages = 3;      // rounds of operands in LDS: the one at hand and two on their way
// The window's rows in the chain's ring, as whole rounds.
__host__ __device__ constexpr uint32_t chain_pad(uint32_t W) { return (W + kRound - 1) / kRound * kRound; }
constexpr uint32_t kQueryWaves = 4;      // wavefronts a block of fbs_layer_query
constexpr uint32_t kListPositions = 512; // positions a block of fbs_layer_lists
constexpr uint32_t kScanQueries = 32;     // queries an item of fbs_layer_scan scores
constexpr uint32_t kNoDrawer = 0xffffffffu;  // the kept drawers of a position that makes no choice
constexpr size_t kLayerLds = 64u << 10;  // LDS bytes a block of these kernels takes at most

}  // namespace

// Each sequence's steps: up to its first token outside the vocabulary (status 1) or to the context's
// end (status 2), whichever comes first, as the step loop refuses them (none for a sequence refused in
// an earlier stretch); the position after them.
__global__ __launch_bounds__(64) void fbs_layer_begin(DevModel M, LayerArgs P) {
  const uint32_t s = blockIdx.x, lane = threadIdx.x;
  if (P.start && P.status[s]) {
    if (lane == 0) P.steps[s] = 0;
    return;
  }
  const uint32_t *tok = P.tokens + (uint64_t)s * P.row + P.start;
  const uint32_t pos = P.in_position ? P.in_position[s] : 0u;
  const uint32_t room = pos < M.context ? M.context - pos : 0u;
  const uint32_t ok = P.len < room ? P.len : room;
  uint32_t first = ok;
  for (uint32_t t = lane; t < ok; t += kWave)
    if (tok[t] >= M.vocab) {
      first = t;
      break;
    }
  first = wave_reduce32(first, OpMin());
  if (lane == 0) {
    P.steps[s] = first;
    P.status[s] = first < ok ? 1 : ok < P.len ? 2 : 0;
    if (P.out_position) P.out_position[s] = pos + first;
  }
}

// Bound by its instructions: 1,413 vector and 358 scalar ones a position and layer at width 256 (most of
// 8 bytes, 5.3 cycles each) take the 448 us that it measures for 152,400 positions.
// The end of layer l - 1 (the output gate on the moved state, rec_out, the feed-forward block; none
// at l = 0, where the position's table row comes in) and the start of layer l (none at l = L), for
// blockIdx.y's sequence, a wavefront a position.
template <int Q>
__global__ __launch_bounds__(64 * kFrontWaves, Q == 1 ? 4 : 2) void fbs_layer_front(DevModel M, LayerArgs P, uint32_t l) {
  extern __shared__ __align__(16) int32_t lds[];
  const uint32_t lane = threadIdx.x % kWave, wave = uniform32(threadIdx.x / kWave);
  uint32_t *seeds = (uint32_t *)lds;
  for (uint32_t i = threadIdx.x; i < kSeedWords; i += blockDim.x)
    seeds[i] = i < kRsqrtSeedWords ? rsqrt_seed_table()[i] : recip_seed_table()[i - kRsqrtSeedWords];
  const Seeds sd(seeds, seeds + kRsqrtSeedWords);
  uint32_t *const keep_lds = (uint32_t *)lds + kSeedWords;  // keep_q31, below 2^31 (layer_model)
  if (threadIdx.x < 16) keep_lds[threadIdx.x] = (uint32_t)M.keep_q31[threadIdx.x];
  // The wave's own: the gather crossbar and the MLP outputs.
  int32_t *const xbar = lds + kSeedWords + 16 + wave * (M.xbar_words + 2 * M.m);
  int64_t *const mlp_out = (int64_t *)(xbar + M.xbar_words);
  __syncthreads();
  const uint32_t s = blockIdx.y, d = M.d, nq = M.nq;
  const uint32_t steps = P.steps[s];
  const bool back = l > 0, front = l < M.L;
  bool qv[Q];
  uint32_t qi[Q], at[Q];
#pragma unroll
  for (int k = 0; k < Q; k++) {
    qi[k] = lane + kWave * k;
    qv[k] = qi[k] < nq;
    at[k] = 4 * (qv[k] ? qi[k] : 0);
  }
  // The layers' tables are read where they are used (from the L1), not held across the wavefront's
  // positions: the registers of a fourth wavefront a SIMD.
  const DevLayer lb = load_layer(M, back ? l - 1 : 0), lf = load_layer(M, front ? l : M.L - 1);
  short4 g_mlp[Q], g_rec[Q];
  uint2 gd_mlp[Q], gd_rec[Q], pw_out[Q], pw_down[Q], pw_rot[Q];
  uint4 pw_rec[Q];
  int4 rbias[Q];
  int32_t dbias[Q], doff[Q];
  uint32_t pw_dec[Q];
  auto load_out = [&]() {
#pragma unroll
    for (int k = 0; k < Q; k++) {
      const uint4 ro = gather8(lb, M.p_rot, k, lane);
      pw_out[k] = make_uint2(ro.z, ro.w);
    }
  };
  auto load_ffn = [&]() {
#pragma unroll
    for (int k = 0; k < Q; k++) {
      g_mlp[k] = gat<short4>(lb.mlp_gain, 2 * at[k]);
      gd_mlp[k] = gat<uint2>(lb.mlp_gain_desc, 2 * at[k]);
    }
  };
  auto load_down = [&]() {
#pragma unroll
    for (int k = 0; k < Q; k++) pw_down[k] = gather4(lb, M.p_down, k, lane);
  };
  auto load_norm = [&]() {
#pragma unroll
    for (int k = 0; k < Q; k++) {
      g_rec[k] = gat<short4>(lf.rec_gain, 2 * at[k]);
      gd_rec[k] = gat<uint2>(lf.rec_gain_desc, 2 * at[k]);
    }
  };
  auto load_rec = [&]() {
#pragma unroll
    for (int k = 0; k < Q; k++) {
      const uint4 rf = gather8(lf, M.p_rot, k, lane);
      pw_rot[k] = make_uint2(rf.x, rf.y);
      pw_rec[k] = gather8(lf, M.p_rec, k, lane);
      pw_dec[k] = gather1(lf, M.p_dec, k, lane);
      rbias[k] = gat<int4>(lf.gate_bias, 4 * (nq + at[k]));
      dbias[k] = gat<int32_t>(lf.gate_bias, at[k]);
      doff[k] = gat<int32_t>(lf.decay_offset, at[k]);
    }
  };
  const uint32_t waves = blockDim.x / kWave;
  uint32_t t = blockIdx.x * P.turns * waves + wave;
#pragma unroll 1
  for (uint32_t i = 0; i < P.turns && t < steps; i++, t += waves) {
    const uint64_t p = (uint64_t)s * P.len + t;
    int32_t x[Q][4];
    if (!back) {
      const uint32_t tok = uniform32(P.tokens[(uint64_t)s * P.row + P.start + t]);
#pragma unroll
      for (int k = 0; k < Q; k++) {
        const uint2 w = qv[k] ? *(const uint2 *)(M.table_b + (uint64_t)tok * d + at[k])
                              : make_uint2(0x80008000u, 0x80008000u);
        const uint32_t ww[2] = {w.x, w.y};
#pragma unroll
        for (int c = 0; c < 4; c++)  // to_exp_i32(v, -12, -16)
          x[k][c] = (int32_t)(int16_t)(uint16_t)(((ww[c >> 1] >> (16 * (c & 1))) & 0xffffu) ^ 0x8000u) << 4;
      }
    } else {
      int4 u4[Q];
      int64_t rhs[Q][4];
#pragma unroll
      for (int k = 0; k < Q; k++) {
        int4 v = *(const int4 *)(P.x + p * d + at[k]);
        u4[k] = *(const int4 *)(P.gate + p * d + at[k]);
        const longlong2 *r = (const longlong2 *)(P.rhs + p * d + at[k]);
        const longlong2 a = r[0], b = r[1];
        rhs[k][0] = a.x, rhs[k][1] = a.y, rhs[k][2] = b.x, rhs[k][3] = b.y;
        if (!qv[k]) v = make_int4(0, 0, 0, 0);
        x[k][0] = v.x, x[k][1] = v.y, x[k][2] = v.z, x[k][3] = v.w;
      }
      // The output gate's product (session.rs:4951-4968), its requantize and rec_out.
      int64_t sc[Q][4], gh[Q][4], gl[Q][4];
      bool fast = true;
      uint64_t mx = 0;
#pragma unroll
      for (int k = 0; k < Q; k++) {
        const int32_t u[4] = {u4[k].x, u4[k].y, u4[k].z, u4[k].w};
        hamilton32_split(u, rhs[k], gh[k], gl[k]);
#pragma unroll
        for (int c = 0; c < 4; c++) fast = fast && (!qv[k] || gate_fast_ok(gh[k][c]));
      }
      if (__all(fast)) {
#pragma unroll
        for (int k = 0; k < Q; k++)
#pragma unroll
          for (int c = 0; c < 4; c++) sc[k][c] = gate_shift14_fast(gh[k][c], gl[k][c]);
      } else {
#pragma unroll
        for (int k = 0; k < Q; k++)
#pragma unroll
          for (int c = 0; c < 4; c++) sc[k][c] = gate_wide14(gh[k][c], gl[k][c]);
      }
#pragma unroll
      for (int k = 0; k < Q; k++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          if (!qv[k]) sc[k][c] = 0;
          mx |= uabs64(sc[k][c]);
        }
      load_out();
      const int32_t bl = wave_bitlen_max(mx);
#pragma unroll
      for (int k = 0; k < Q; k++)
        if (qv[k]) requant_publish(xbar, 4 * qi[k], sc[k], bl);
      wave_sync();
#pragma unroll
      for (int k = 0; k < Q; k++)
        if (qv[k])
#pragma unroll
          for (int c = 0; c < 4; c++)
            x[k][c] = sat_add32(x[k][c], gather(xbar, c < 2 ? pw_out[k].x : pw_out[k].y, c & 1));
      wave_sync();
      // The feed-forward block (session.rs:4005-4025).
      load_ffn();
      norm_publish<Q>(M, sd, x, qv, qi, g_mlp, gd_mlp, xbar);
      wave_sync();
      uint64_t mmx = 0;
#pragma unroll 1
      for (uint32_t j = 0; j < M.mpl; j++) {
        const uint32_t mq = lane + kWave * j;
        const uint4 pw = gather8(lb, M.p_mlp, j, lane);
        int32_t gq[4], up[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
          gq[c] = gather(xbar, c < 2 ? pw.x : pw.y, c & 1);
          up[c] = gather(xbar, c < 2 ? pw.z : pw.w, c & 1);
        }
        if (mq < M.nm) {
          int64_t mo[4];
          mlp_gate(M, sd, gq, up, mo);
          longlong2 *o = (longlong2 *)(mlp_out + 4 * mq);
          o[0] = make_longlong2(mo[0], mo[1]);
          o[1] = make_longlong2(mo[2], mo[3]);
#pragma unroll
          for (int c = 0; c < 4; c++) mmx |= uabs64(mo[c]);
        }
      }
      load_down();
      const int32_t mbl = wave_bitlen_max(mmx);
      wave_sync();
#pragma unroll 1
      for (uint32_t j = 0; j < M.mpl; j++) {
        const uint32_t mq = lane + kWave * j;
        if (mq < M.nm) {
          const longlong2 *o = (const longlong2 *)(mlp_out + 4 * mq);
          const longlong2 a = o[0], b = o[1];
          const int64_t v[4] = {a.x, a.y, b.x, b.y};
          requant_publish(xbar, 4 * mq, v, mbl);
        }
      }
      wave_sync();
#pragma unroll
      for (int k = 0; k < Q; k++)
        if (qv[k])
#pragma unroll
          for (int c = 0; c < 4; c++)
            x[k][c] = sat_add32(x[k][c], gather(xbar, c < 2 ? pw_down[k].x : pw_down[k].y, c & 1));
      wave_sync();
    }
#pragma unroll
    for (int k = 0; k < Q; k++)
      if (qv[k]) *(int4 *)(P.x + p * d + at[k]) = make_int4(x[k][0], x[k][1], x[k][2], x[k][3]);
    if (front) {
      load_norm();
      norm_publish<Q>(M, sd, x, qv, qi, g_rec, gd_rec, xbar);
      load_rec();
      wave_sync();
#pragma unroll
      for (int k = 0; k < Q; k++) {
        if (!qv[k]) continue;
        const int32_t rb[4] = {rbias[k].x, rbias[k].y, rbias[k].z, rbias[k].w};
        int32_t rot[4], gv[4], dr[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
          dr[c] = gather(xbar, c < 2 ? pw_rec[k].x : pw_rec[k].y, c & 1);
          gv[c] = gather(xbar, c < 2 ? pw_rec[k].z : pw_rec[k].w, c & 1);
          rot[c] = sat_add32(gather(xbar, c < 2 ? pw_rot[k].x : pw_rot[k].y, c & 1), rb[c]);
        }
        const int32_t dec = sat_add32(gather(xbar, pw_dec[k], 0), dbias[k]);
        // Lane weights (session.rs:4989-5026), the transition's rotation and the output gate.
        int32_t sq = sat_add32(dec, doff[k]);
        sq = sq < 0 ? 0 : sq > 65536 ? 65536 : sq;
        uint32_t idx = (uint32_t)sq >> 12;
        idx = idx > 15 ? 15 : idx;
        int32_t u[4];
        wave_unit_q30(rot, kRotationEps, u, sd);
        *(int4 *)(P.turn + p * d + at[k]) = make_int4(u[0] >> idx, u[1] >> idx, u[2] >> idx, u[3] >> idx);
        P.keep[p * nq + qi[k]] = keep_lds[idx];
        wave_unit_q30(gv, kGateEps, u, sd);
        *(int4 *)(P.gate + p * d + at[k]) = make_int4(u[0], u[1], u[2], u[3]);
        *(int4 *)(P.drive + p * d + at[k]) = make_int4(dr[0], dr[1], dr[2], dr[3]);
      }
      wave_sync();
    }
  }
}

// Layer l's windows (session.rs:4842-4868) and transport (session.rs:5097-5145) for blockIdx.y's
// sequence, a lane a channel, in rounds of 8 positions: wavefront 1 sums a round's windows into LDS while
// wavefront 0 moves the state through the round before and writes it at the residual's exponent. What a
// round reads comes into LDS by direct loads two rounds ahead:
// the drives into a ring of the window and three rounds, the transitions and keeps for wavefront 0.
// - Windows: tap k's word and a row serve eight positions; the positions' rows lie in registers and move
//   one place a tap, by naming and not by moving in eight taps.
// - Transport: the four lanes of a quaternion exchange its halves by DPP: component k of T (x) b is the
//   sum over i of +-T_i b_(k xor i), so a lane makes four products of each half and not the sixteen
//   of a whole quaternion. Eight positions move by transport_fast's form without a branch; where one
//   left its ranges, they move again from the state before them in 128 bits.
// Lanes past the width repeat the last quaternion's.
// 300 sequences of 508 positions, width 256: 214 us. Its bytes, 17 a channel and position, take 130 at 5
// TB/s; five blocks a CU (their LDS) leave a SIMD two or three wavefronts, whose rounds wait for one
// another. Windows in a kernel of their own (their sums through memory): 360; operands asked for one
// round ahead: 258.
// Form: the layer's tap words.
enum Taps : int {
  kTapsHigh,  // tap_word's, every one of which times 16 fits 32 bits (P.taps_high)
  kTapsWord,  // tap_word's
  kTapsPair,  // tap_pair's
};
template <Taps Form>
__global__ __launch_bounds__(64 * kChainWaves, 2) void fbs_layer_chain(DevModel M, LayerArgs P, uint32_t l) {
  extern __shared__ __align__(16) int32_t lds[];
  const uint32_t lane = threadIdx.x % kWave, wave = uniform32(threadIdx.x / kWave), k = lane % 4;
  const uint32_t s = blockIdx.y, d = M.d, nq = M.nq, L = M.L, W = M.W;
  const uint32_t ch0 = blockIdx.x * kWave;
  const uint32_t lv = ch0 + lane < d ? lane : d - 4 - ch0 + k, ch = ch0 + lv;
  const uint32_t steps = P.steps[s];
  const uint64_t p0 = (uint64_t)s * P.len;
  const int32_t *const drive = P.drive + p0 * d;
  const int32_t *const turn = P.turn + p0 * d;
  const uint32_t *const keeps = P.keep + p0 * nq;
  const int32_t *const before = P.in_history ? P.in_history + ((uint64_t)s * L + l) * W * d : nullptr;
  const uint32_t pad = chain_pad(W), ring_rows = pad + kStages * kRound;
  int64_t (*const sums)[kRound][kWave] = (int64_t(*)[kRound][kWave])lds;   // [2]
  int32_t (*const turns)[kRound][kWave] = (int32_t(*)[kRound][kWave])(sums + 2);  // [kStages]
  uint32_t (*const kept)[kRound][16] = (uint32_t(*)[kRound][16])(turns + kStages);  // [kStages]
  int32_t (*const taps)[kWave] = (int32_t(*)[kWave])(kept + kStages);   // [W + 1]
  int32_t (*const ring)[kWave] = taps + W + 1;                    // [ring_rows]: position t at (t + pad) mod ring_rows

  // Round r's rows of `src` (a row a position) to dst, four rows a load: lane 16 i + j brings piece j of
  // row i; rows past the last position and pieces past the width repeat them.
  const auto bring = [&](const int32_t *src, uint32_t r, int32_t (*dst)[kWave]) {
    const uint32_t c = ch0 + 4 * (lane % 16), cc = c < d ? c : d - 4;
#pragma unroll
    for (uint32_t j = 0; j < kRound / 4; j++) {
      uint32_t t = r * kRound + 4 * j + lane / 16;
      t = t < steps ? t : steps - 1;
      __builtin_amdgcn_global_load_lds((global_void *)(src + (uint64_t)t * d + cc), (lds_void *)dst[4 * j], 16, 0, 0);
    }
  };
  const auto bring_keeps = [&](uint32_t r, uint32_t stage) {
    if (lane >= 4 * kRound) return;
    uint32_t t = r * kRound + lane / 4;
    t = t < steps ? t : steps - 1;
    const uint32_t q = ch0 / 4 + 4 * (lane % 4), qq = q < nq ? q : nq - 4;
    __builtin_amdgcn_global_load_lds((global_void *)(keeps + (uint64_t)t * nq + qq), (lds_void *)kept[stage], 16, 0, 0);
  };
  // The ring's place of round r's first row: (8 r + pad) mod ring_rows, kept as the rounds go.
  const int32_t bias = gat<int32_t>(load_layer(M, l).conv_bias, 4 * ch);
  const auto windows = [&](uint32_t r, uint32_t place) {
    int64_t acc[kRound];
    int32_t rows[kRound];  // at tap i, position t0 + u's row t0 + u - i is rows[(u - i) mod kRound]
#pragma unroll
    for (uint32_t u = 0; u < kRound; u++) acc[u] = bias, rows[u] = ring[place + u][lv];
    uint32_t back = place;
#pragma unroll 1
    for (uint32_t i0 = 0; i0 <= W; i0 += kRound) {
      int32_t tap[kRound], next[kRound];
      back = (back ? back : ring_rows) - kRound;  // the ring holds whole rounds: eight rows do not wrap
#pragma unroll
      for (uint32_t j = 0; j < kRound; j++) {
        const int32_t t = taps[i0 + j < W ? i0 + j : W][lv];
        tap[j] = Form == kTapsHigh ? t << 4 : t;
        next[j] = ring[back + kRound - 1 - j][lv];
      }
#pragma unroll
      for (uint32_t j = 0; j < kRound; j++) {
        if (i0 + j > W) break;
#pragma unroll
        for (uint32_t u = 0; u < kRound; u++) {
          const int32_t v = rows[(u + kRound - j) % kRound];
          if constexpr (Form == kTapsHigh) {
            // tap_word_apply with the word times 16: the floor is the sum's high half.
            const uint32_t half = (1u << 31) + (uint32_t)(tap[j] >> 31);
            const int32_t term = (int32_t)(((int64_t)v * tap[j] + (int64_t)(uint64_t)half) >> 32);
            uint64_t carry;
            asm("v_mad_i64_i32 %0, %1, %2, 1, %0" : "+v"(acc[u]), "=s"(carry) : "v"(term));
          } else {
            acc[u] = wadd64(acc[u], Form == kTapsWord ? tap_word_apply(v, tap[j]) : tap_pair_apply(v, tap[j]));
          }
        }
        // The last position's row leaves, the one before the first's enters in its place.
        rows[kRound - 1 - j] = next[j];
      }
    }
#pragma unroll
    for (uint32_t u = 0; u < kRound; u++) sums[r & 1][u][lane] = acc[u];
  };

  int64_t *const out = P.rhs + p0 * d;
  // The signs of T_1..T_3 in component k: masks and their negations.
  const int32_t s1 = k == 0 || k == 2 ? -1 : 0, s2 = k == 0 || k == 3 ? -1 : 0, s3 = k < 2 ? -1 : 0;
  const int32_t n1 = -s1, n2 = -s2, n3 = -s3;
  int64_t h = wave == 0 && P.in_state ? P.in_state[((uint64_t)s * L + l) * d + ch] : 0;
  // Round r's positions (full: all kRound of them).
  const auto move = [&](auto full, uint32_t r, uint32_t stage) {
    const uint32_t t0 = r * kRound;
    const uint32_t n = full ? kRound : steps - t0;
    const int64_t h0 = h;
    int64_t hn = h;
    uint32_t out_h = 0, out_w = 0;  // bits 28.. and 14..: a product or a window sum past transport_fast's ranges
    if (__all(split_ok(h))) {
      int4 T8[kRound];
      uint32_t keep8[kRound];
      int64_t w[kRound];
#pragma unroll
      for (uint32_t i = 0; i < kRound; i++) {
        T8[i] = *(const int4 *)&turns[stage][i][lv & ~3u];
        keep8[i] = kept[stage][i][lv / 4];
        w[i] = sums[r & 1][i][lv];
      }
#pragma unroll
      for (uint32_t i = 0; i < kRound; i++) {
        const int4 T = T8[i];
        const int32_t a1 = (T.y ^ s1) + n1, a2 = (T.z ^ s2) + n2, a3 = (T.w ^ s3) + n3;
        const uint32_t hi = (uint32_t)(((uint64_t)h + (1ull << 31)) >> 32), lo = (uint32_t)h;
        const int32_t wh = (int32_t)(w[i] >> 32), keep = (int32_t)keep8[i];
        const uint64_t K = (uint64_t)keep8[i] * (uint32_t)w[i];
        uint32_t z0 = (((uint32_t)K & 0x7fffu) << 16) + (1u << 30);
        asm("" : "+v"(z0));  // added as 32 bits, not again as 64
        const int64_t H = (int64_t)T.x * (int32_t)hi + (int64_t)a1 * (int32_t)dpp32<0xB1>(hi) +
                          (int64_t)a2 * (int32_t)dpp32<0x4E>(hi) + (int64_t)a3 * (int32_t)dpp32<0x1B>(hi);
        const int64_t Z = (int64_t)(uint64_t)z0 + (int64_t)T.x * (int32_t)lo + (int64_t)a1 * (int32_t)dpp32<0xB1>(lo) +
                          (int64_t)a2 * (int32_t)dpp32<0x4E>(lo) + (int64_t)a3 * (int32_t)dpp32<0x1B>(lo);
        out_h |= (uint32_t)(H >> 32) + (1u << 27);
        out_w |= (uint32_t)wh + (1u << 13);
        // transport_fast(H, L, keep, wide)
        h = (int64_t)(((uint64_t)(H + (int64_t)keep * (int32_t)((uint32_t)wh << 16)) << 1) + (K >> 15)) + (Z >> 31);
        if (i < n) hn = h, out[(uint64_t)(t0 + i) * d + ch] = (h + (1ll << 15)) >> 16;  // |h| < 2^62: no saturation
      }
      h = hn;
      if (!__any((out_h >> 28) | (out_w >> 14))) return;
    }
    h = h0;
#pragma unroll 1
    for (uint32_t i = 0; i < n; i++) {
      const int4 T = *(const int4 *)&turns[stage][i][lv & ~3u];
      const uint64_t v = (uint64_t)h;
      const int32_t a[4] = {T.x, T.y, T.z, T.w};
      const int64_t hq[4] = {(int64_t)dpp64<0x00>(v), (int64_t)dpp64<0x55>(v), (int64_t)dpp64<0xAA>(v),
                             (int64_t)dpp64<0xFF>(v)};
      int64_t H[4], Lo[4];
      hamilton32_hl(a, hq, H, Lo);
      const int64_t hk = k == 0 ? H[0] : k == 1 ? H[1] : k == 2 ? H[2] : H[3];
      const int64_t lk = k == 0 ? Lo[0] : k == 1 ? Lo[1] : k == 2 ? Lo[2] : Lo[3];
      const u128 term = (u128)((i128)(uint64_t)kept[stage][i][lv / 4] * (i128)sums[r & 1][i][lv]) << 16;
      h = shift_wide((i128)((u128)(((i128)hk << 32) + (i128)lk) + term), 31);  // transport_wide
      out[(uint64_t)(t0 + i) * d + ch] = shift(h, kResidualExp - kStateExp);
    }
  };

  const uint32_t rounds = (steps + kRound - 1) / kRound;
  if (steps) {
    if (wave == 1) {
      bring(drive, 0, ring + pad);
      for (uint32_t r = 1; r < kStages && r < rounds; r++) bring(drive, r, ring + pad + r * kRound);
      for (uint32_t r = 0; r < kStages - 1 && r < rounds; r++) {
        bring(turn, r, turns[r]);
        bring_keeps(r, r);
      }
    }
    const uint32_t c = ch0 + 4 * (lane % 16), cc = c < d ? c : d - 4;
    for (uint32_t i0 = 4 * wave; i0 <= W; i0 += 4 * kChainWaves) {
      const uint32_t i = i0 + lane / 16;
      if (i <= W)
        __builtin_amdgcn_global_load_lds((global_void *)(M.tap_words + ((uint64_t)l * (W + 1) + i) * d + cc),
                                         (lds_void *)taps[i0], 16, 0, 0);
    }
    // The session's rows before the first position (row r at place pad - 1 - r; the places of rows past the
    // window are never used); none: zero rows, whose terms are 0.
    for (uint32_t i0 = 4 * wave; i0 < pad; i0 += 4 * kChainWaves) {
      const uint32_t i = i0 + lane / 16, r = pad - 1 - i;
      if (!before)
        *(int4 *)&ring[i][4 * (lane % 16)] = make_int4(0, 0, 0, 0);
      else if (r < W)
        __builtin_amdgcn_global_load_lds((global_void *)(before + (uint64_t)r * d + cc), (lds_void *)ring[i0], 16, 0, 0);
    }
    wait_lds_dma();
    pair_sync();
    if (wave) windows(0, pad);
  }
  // A loop a wavefront: in one, the compiler would have wavefront 0's LDS reads wait for the direct loads of
  // wavefront 1's branch and with them for its own stores.
  if (wave == 0) {
    uint32_t stage = 0;
    for (uint32_t r = 0; r < rounds; r++) {
      pair_sync();  // round r's sums, transitions and keeps are there
      if ((r + 1) * kRound <= steps)
        move(std::true_type(), r, stage);
      else
        move(std::false_type(), r, stage);
      stage = stage + 1 == kStages ? 0 : stage + 1;
    }
  } else {
    uint32_t place = pad, stage = 0;  // of round r's rows in the ring and of its transitions
    for (uint32_t r = 0; r < rounds; r++) {
      pair_sync();  // round r - 1's sums and transitions have been read
      if (r + 1 == rounds) break;
      const uint32_t next = place + kRound == ring_rows ? 0 : place + kRound;
      // Into the places of round r - 1's transitions and of rows that no window reads any more.
      if (r + kStages - 1 < rounds) {
        const uint32_t last = stage ? stage - 1 : kStages - 1;
        bring(turn, r + kStages - 1, turns[last]);
        bring_keeps(r + kStages - 1, last);
      }
      if (r + kStages < rounds) {
        const uint32_t to = place + kStages * kRound;
        bring(drive, r + kStages, ring + (to >= ring_rows ? to - ring_rows : to));
      }
      windows(r + 1, next);
      // What this round asked for (2 kRound / 4 + 1 loads) may still be on its way.
      static_assert(kRound == 8, "the count below");
      if (r + kStages < rounds)
        __builtin_amdgcn_s_waitcnt(0x0f75);  // vmcnt(5)
      else
        wait_lds_dma();
      place = next;
      stage = stage + 1 == kStages ? 0 : stage + 1;
    }
  }
  if (steps < P.len || !P.out_state) return;  // a refused sequence exports nothing
  if (wave == 0) {
    P.out_state[((uint64_t)s * L + l) * d + ch] = h;
  } else if (wave == 1) {
    // Row r is the drive r + 1 positions back; the oldest first, so that the rows may be the ones that
    // came in (all of them have been read).
    int32_t *const rows = P.out_history + ((uint64_t)s * L + l) * W * d;
    for (int32_t r = (int32_t)W - 1; r >= 0; r--) {
      int32_t v = 0;
      if ((uint32_t)r < P.len)
        v = drive[(uint64_t)(P.len - 1 - r) * d + ch];
      else if (before)
        v = before[(uint64_t)(r - P.len) * d + ch];
      rows[(uint64_t)r * d + ch] = v;
    }
  }
}

// The final norm, the Q12 query and the drawer selection of A.n positions from P.first on, a wavefront
// each in turn: the position's query for the scan (RunArgs::job_query) and its kept drawers. (32,768 of
// width 256 among 256 drawers 59 us, and 15 for their lists; a block a position that entered the lists
// itself 185: eight atomics with a result a position.)
template <int Q, bool T8>
__global__ __launch_bounds__(64 * kQueryWaves) void fbs_layer_query(DevModel M, LayerArgs P, RunArgs A) {
  extern __shared__ __align__(16) int32_t lds[];
  const uint32_t lane = threadIdx.x % kWave, wave = uniform32(threadIdx.x / kWave), d = M.d;
  uint32_t *seeds = (uint32_t *)lds;
  for (uint32_t i = threadIdx.x; i < kSeedWords; i += blockDim.x)
    seeds[i] = i < kRsqrtSeedWords ? rsqrt_seed_table()[i] : recip_seed_table()[i - kRsqrtSeedWords];
  const Seeds sd(seeds, seeds + kRsqrtSeedWords);
  int32_t *const query = lds + kSeedWords + wave * (d + kMaxProbes + ((M.D + 3u) & ~3u));
  uint32_t *const kept = (uint32_t *)(query + d), *const dscore = kept + kMaxProbes;
  __syncthreads();
  bool qv[Q];
  uint32_t qi[Q];
  short4 g[Q];
  uint2 gd[Q];
#pragma unroll
  for (int k = 0; k < Q; k++) {
    qi[k] = lane + kWave * k;
    qv[k] = qi[k] < M.nq;
    const uint32_t at = 4 * (qv[k] ? qi[k] : 0);
    g[k] = *(const short4 *)(M.final_gain + at);
    gd[k] = *(const uint2 *)(M.final_gain_desc + at);
  }
  const uint32_t waves = blockDim.x / kWave;
  for (uint32_t i = blockIdx.x * waves + wave; i < A.n; i += gridDim.x * waves) {
    const uint32_t p = P.first + i;
    uint32_t s = (uint32_t)((p * P.len_recip) >> 32);  // p / len, or one less
    uint32_t t = p - s * P.len;
    if (t >= P.len) s++, t -= P.len;
    s = uniform32(s), t = uniform32(t);
    if (t >= P.steps[s] || (!P.out_tokens && P.start + t + 1 == P.row)) {
      if (lane < M.P) P.kept[(uint64_t)i * M.P + lane] = kNoDrawer;
      continue;
    }
    const uint64_t at_row = (uint64_t)s * P.row + P.start + t;  // its place in the rows
    int32_t x[Q][4];
#pragma unroll
    for (int k = 0; k < Q; k++) {
      int4 v = *(const int4 *)(P.x + (uint64_t)p * d + 4 * (qv[k] ? qi[k] : 0));
      if (!qv[k]) v = make_int4(0, 0, 0, 0);
      x[k][0] = v.x, x[k][1] = v.y, x[k][2] = v.z, x[k][3] = v.w;
    }
    int64_t v[Q][4];
    norm_gain<Q>(M, sd, x, g, gd, v);
#pragma unroll
    for (int k = 0; k < Q; k++)
      if (qv[k]) {
        int32_t qa[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const int32_t y = to_exp_i32(v[k][c], kNormFineExp, kQ12Exp);
          qa[c] = y > 32767 ? 32767 : y < -32768 ? -32768 : y;
        }
        const int4 qq = make_int4(qa[0], qa[1], qa[2], qa[3]);
        *(int4 *)(query + 4 * qi[k]) = qq;
        if (P.out_query) *(int4 *)(P.out_query + at_row * d + 4 * qi[k]) = qq;
      }
    wave_sync();
    uint32_t b, e;
    writer_select(M, query, dscore, kept, lane, b, e);
    if (lane < M.P) {
      P.kept[(uint64_t)i * M.P + lane] = kept[lane];
      if (P.out_kept) P.out_kept[at_row * M.P + lane] = kept[lane];
    }
    job_words<Q, T8>(M, A, i, query, qv, qi);
    if (lane == 0) {
      A.job_best[i] = ~0ull;
      A.job_flag[i] = 1u;
    }
    wave_sync();
  }
}

// The drawers' lists of the positions that kept them, and the scan's work items. A block counts its
// positions' drawers in LDS and takes their places with one atomic a drawer: one a position and drawer
// met at the few large drawers of skewed sizes. The block that takes a slice's first place opens its
// items.
__global__ __launch_bounds__(256) void fbs_layer_lists(DevModel M, LayerArgs P, RunArgs A) {
  extern __shared__ uint32_t places[];  // a drawer's count, then its next place
  const uint32_t i0 = blockIdx.x * kListPositions;
  const uint32_t n = A.n - i0 < kListPositions ? A.n - i0 : kListPositions;
  const uint32_t *const kept = P.kept + (uint64_t)i0 * M.P;
  for (uint32_t c = threadIdx.x; c < M.D; c += blockDim.x) places[c] = 0;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
    for (uint32_t j = 0; j < M.P; j++) {
      const uint32_t c = kept[i * M.P + j];
      if (c != kNoDrawer) atomicAdd(places + c, 1u);
    }
  __syncthreads();
  for (uint32_t c = threadIdx.x; c < M.D; c += blockDim.x) {
    const uint32_t m = places[c];
    if (m == 0) continue;
    const uint32_t at = atomicAdd(A.drawer_count + c, m);
    places[c] = at;
    const uint32_t b = M.offsets[c], e = M.offsets[c + 1];
    const uint32_t chunks = (e - b + kServeRows - 1) / kServeRows;
    const uint32_t g0 = (at + kScanQueries - 1) / kScanQueries, g1 = (at + m + kScanQueries - 1) / kScanQueries;
    if (g0 >= g1 || chunks == 0) continue;
    uint32_t i = atomicAdd(A.item_count, (g1 - g0) * chunks);
    for (uint32_t g = g0; g < g1; g++)
      for (uint32_t m0 = b; m0 < e; m0 += kServeRows, i++)
        if (i < A.item_cap)
          A.items[i] = make_uint4(m0, e - m0 < kServeRows ? e - m0 : kServeRows, c * A.list_stride + g * kScanQueries, c);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
    for (uint32_t j = 0; j < M.P; j++) {
      const uint32_t c = kept[i * M.P + j];
      if (c == kNoDrawer) continue;
      const uint32_t at = atomicAdd(places + c, 1u);
      if (at < A.list_stride) A.drawer_list[(uint64_t)c * A.list_stride + at] = i0 + i;
    }
}

// The scan of fbs_serve.hip for many queries: the blocks (a wavefront each) take the items in turn, and an
// item scores up to 64 member rows of a drawer against a slice of 32 of the queries that kept it,
// staged in LDS. Lane 16 g + r holds rows r, r + 16, r + 32 and r + 48 and scores them against queries
// g, g + 4, ... of the slice: so a 16-byte read of a query (one address a row of 16 lanes) serves 16
// SADs, and a query's lowest (L1, token) is a reduction over 16 lanes. fbs_serve_scan, a row a lane and
// every query in all lanes, reads 16 bytes for 4 SADs and reduces 64 lanes a query, a third of its
// instructions: 32,768 queries of width 256 that kept 8 of 256 drawers 433 us, here 310. One-token
// launches keep it: their thousand queries fill few slices of 32, and a wavefront then waits through
// four segments of a row one after another (1,024 sessions 2.88 ms per 32 tokens, with this 3.09).
// Queries in lanes' registers and rows by scalar loads: 529 us, the scalar cache missing on every row.
// RW: the row words (biased 16-bit pairs) of a segment; rows of more words are scored in segments of
// RW, the sums carried across. T8: an int8 table, whose rows (code + 128 bytes) widen at the SADs as the
// fused writer's scan widens them (widen8), against queries in that scan's scaled form.
template <int RW, bool T8>
__global__ __launch_bounds__(64, 2) void fbs_layer_scan(DevModel M, ServeScan J) {
  constexpr uint32_t kRows = kServeRows / 16;          // rows a lane
  constexpr uint32_t kSets = kScanQueries / 4;       // sessions a lane
  constexpr uint32_t kQuads = RW / 4;                  // 16-byte pieces of a query's segment
  constexpr uint32_t kStage = kScanQueries * kQuads / kWave;
  constexpr uint32_t kRowQuads = T8 ? RW / 8 : RW / 4;
  __shared__ __align__(16) uint32_t qs[kScanQueries * RW];
  const uint32_t lane = threadIdx.x, r16 = lane % 16, set = lane / 16;
  uint32_t total = uniform32(J.item_count[0]);
  total = total < J.item_cap ? total : J.item_cap;
  const uint32_t words = M.d / 2;
  for (uint32_t it = blockIdx.x; it < total; it += gridDim.x) {
    const uint4 item = J.items[it];
    const uint32_t beg = uniform32(item.x), rows = uniform32(item.y);
    const uint32_t lbeg = uniform32(item.z), c = uniform32(item.w);
    uint32_t nc = uniform32(J.drawer_count[c]);
    nc = nc < J.list_stride ? nc : J.list_stride;  // a list holds at most list_stride sessions
    const uint32_t g = lbeg - c * J.list_stride;
    if (g >= nc) continue;
    const uint32_t ns = nc - g < kScanQueries ? nc - g : kScanQueries;
    const uint32_t *list = J.drawer_list + lbeg;
    uint32_t tok[kRows];
    const uint4 *row[kRows];
#pragma unroll
    for (uint32_t m = 0; m < kRows; m++) {
      const uint32_t k = r16 + 16 * m;
      tok[m] = M.members[beg + (k < rows ? k : 0)];
      row[m] = T8 ? (const uint4 *)(M.table8 + (uint64_t)tok[m] * M.d)
                  : (const uint4 *)((const uint32_t *)M.table_b + (uint64_t)tok[m] * words);
    }
    // The query quads this lane stages: piece (lane + 64 j) % kQuads of session (lane + 64 j) / kQuads.
    uint32_t stage_sid[kStage];
#pragma unroll
    for (uint32_t j = 0; j < kStage; j++) {
      const uint32_t i = (lane + kWave * j) / kQuads;
      stage_sid[j] = list[i < ns ? i : 0];
    }
    uint32_t acc[kSets][kRows];
#pragma unroll
    for (uint32_t j = 0; j < kSets; j++)
#pragma unroll
      for (uint32_t m = 0; m < kRows; m++) acc[j][m] = 0;
#pragma unroll 1
    for (uint32_t seg = 0; seg < words; seg += RW) {
      // Once the last segment's (or item's) reads are done: the sessions' query words of this
      // segment go to LDS by direct loads (no registers), the rows' words to registers, every
      // load issued before the first is waited for.
      wave_sync();
#pragma unroll
      for (uint32_t j = 0; j < kStage; j++)
        if (kWave * j < ns * kQuads)
          __builtin_amdgcn_global_load_lds(
              (global_void *)(J.job_query + (uint64_t)stage_sid[j] * words + seg + 4 * (lane % kQuads)),
              (lds_void *)(qs + 4 * kWave * j), 16, 0, 0);
      uint4 r[kRows][kRowQuads];
#pragma unroll
      for (uint32_t m = 0; m < kRows; m++)
#pragma unroll
        for (uint32_t w = 0; w < kRowQuads; w++) r[m][w] = row[m][(T8 ? seg / 8 : seg / 4) + w];
      wait_lds_dma();
      // Eight sessions at a time (two a lane), as many as the slice holds; sessions past ns read words
      // never staged and are not used.
#pragma unroll
      for (uint32_t j0 = 0; j0 < kSets; j0 += 2) {
        if (4 * j0 < ns) {
#pragma unroll
          for (uint32_t w = 0; w < kQuads; w++) {
            uint4 x[kRows];  // the rows' words against the queries' piece w
#pragma unroll
            for (uint32_t m = 0; m < kRows; m++) {
              if constexpr (T8) {
                const uint4 p = r[m][w / 2];
                widen8(w % 2 ? p.z : p.x, x[m].x, x[m].y);
                widen8(w % 2 ? p.w : p.y, x[m].z, x[m].w);
              } else {
                x[m] = r[m][w];
              }
            }
#pragma unroll
            for (uint32_t j = j0; j < j0 + 2; j++) {
              const uint4 q = *(const uint4 *)(qs + (4 * j + set) * RW + 4 * w);
#pragma unroll
              for (uint32_t m = 0; m < kRows; m++) {
                uint32_t a = acc[j][m];
                a = sad2_u16(q.x, x[m].x, a);
                a = sad2_u16(q.y, x[m].y, a);
                a = sad2_u16(q.z, x[m].z, a);
                a = sad2_u16(q.w, x[m].w, a);
                acc[j][m] = a;
              }
            }
          }
        }
      }
    }
    // Lane 16 g + j takes session 4 j + g.
    uint64_t mine = ~0ull;
#pragma unroll
    for (uint32_t j = 0; j < kSets; j++) {
      if (4 * j < ns) {
        uint64_t v = ~0ull;
#pragma unroll
        for (uint32_t m = 0; m < kRows; m++) {
          const uint64_t o = ((uint64_t)acc[j][m] << 32) | tok[m];
          v = r16 + 16 * m < rows && o < v ? o : v;
        }
        v = row16_min(v);
        mine = r16 == j ? v : mine;
      }
    }
    const uint32_t i = 4 * r16 + set;
    if (r16 < kSets && i < ns) atomicMin(J.job_best + list[i], (unsigned long long)mine);
  }
}

// The stretch's choices to the rows' place and their matches with the rows' next tokens. The choices may go
// over the rows themselves, as a step's choice goes over its own token: a round's next tokens are read
// before any of its choices is written.
__global__ __launch_bounds__(256) void fbs_layer_choices(LayerArgs P) {
  const uint32_t s = blockIdx.x;
  const uint32_t steps = P.steps[s];
  const uint32_t *tok = P.tokens + (uint64_t)s * P.row + P.start;
  uint32_t hits = 0;
  for (uint32_t t0 = 0; t0 < steps; t0 += blockDim.x) {
    const uint32_t t = t0 + threadIdx.x;
    const bool in = t < steps, next = in && P.start + t + 1 < P.row;
    const uint32_t after = next ? tok[t + 1] : 0;
    const uint32_t c = next || (in && P.out_tokens) ? P.chosen[(uint64_t)s * P.len + t] : 0;
    if (P.out_tokens) {
      __syncthreads();
      if (in) P.out_tokens[(uint64_t)s * P.row + P.start + t] = c;
    }
    hits += next && c == after;
  }
  hits = wave_reduce32(hits, OpAdd());
  if (P.matches && threadIdx.x % kWave == 0 && hits) atomicAdd(P.matches, (unsigned long long)hits);
}

namespace {

hipError_t run_kernel(const void *f, dim3 grid, uint32_t threads, void **args, size_t lds, hipStream_t st) {
  const hipError_t e = hipLaunchKernel(f, grid, dim3(threads), args, lds, st);
  return e != hipSuccess ? e : hipGetLastError();
}

size_t front_lds(const DevModel &M, uint32_t waves) { return 4ull * (kSeedWords + 16 + waves * (M.xbar_words + 2 * M.m)); }
size_t chain_lds(const DevModel &M) {
  return 4ull * kWave * (4 * kRound + kStages * (kRound + kRound / 4 + kRound) + M.W + 1 + chain_pad(M.W));
}
size_t query_lds(const DevModel &M, uint32_t waves) {
  return 4ull * (kSeedWords + waves * (M.d + kMaxProbes + ((M.D + 3u) & ~3u)));
}

// The front and query kernels' wavefronts a block: four, or fewer where wide layers' crossbars or many
// drawers' scores need the room.
uint32_t front_waves(const DevModel &M) {
  for (uint32_t w = kFrontWaves; w > 0; w /= 2)
    if (front_lds(M, w) <= kLayerLds) return w;
  return 0;
}
uint32_t query_waves(const DevModel &M) {
  for (uint32_t w = kQueryWaves; w > 0; w /= 2)
    if (query_lds(M, w) <= kLayerLds) return w;
  return 0;
}

}  // namespace

bool fbs_layers_fit(const DevModel &M) {
  return front_waves(M) != 0 && query_waves(M) != 0 && chain_lds(M) <= kLayerLds;
}

hipError_t launch_fbs_layers(const DevModel &M, const LayerArgs &P, bool rows, hipStream_t stream) {
  DevModel m = M;
  LayerArgs p = P;
  uint32_t l = 0;
  void *args[] = {&m, &p, &l};
  hipError_t e = run_kernel((const void *)fbs_layer_begin, dim3(P.n), kWave, args, 0, stream);
  const void *front = M.qpl == 1   ? (const void *)fbs_layer_front<1>
                      : M.qpl == 2 ? (const void *)fbs_layer_front<2>
                                   : (const void *)fbs_layer_front<4>;
  const uint32_t waves = front_waves(M), per = waves * P.turns;
  for (l = 0; l < M.L + (rows ? 1u : 0u) && e == hipSuccess; l++) {
    e = run_kernel(front, dim3((P.len + per - 1) / per, P.n), kWave * waves, args, front_lds(M, waves), stream);
    if (l == M.L) break;
    const void *chain = (M.tap_pairs >> l) & 1 ? (const void *)fbs_layer_chain<kTapsPair>
                        : P.taps_high          ? (const void *)fbs_layer_chain<kTapsHigh>
                                               : (const void *)fbs_layer_chain<kTapsWord>;
    if (e == hipSuccess)
      e = run_kernel(chain, dim3((M.d + kWave - 1) / kWave, P.n), kWave * kChainWaves, args, chain_lds(M), stream);
  }
  return e;
}

hipError_t launch_fbs_layer_query(const DevModel &M, const LayerArgs &P, const RunArgs &A, const ServeScan &S,
                                  uint32_t cus, hipStream_t stream) {
  DevModel m = M;
  LayerArgs p = P;
  RunArgs a = A;
  const bool t8 = M.table8 != nullptr;
  const void *f = M.qpl == 1 ? (t8 ? (const void *)fbs_layer_query<1, true> : (const void *)fbs_layer_query<1, false>)
                  : M.qpl == 2
                      ? (t8 ? (const void *)fbs_layer_query<2, true> : (const void *)fbs_layer_query<2, false>)
                      : (t8 ? (const void *)fbs_layer_query<4, true> : (const void *)fbs_layer_query<4, false>);
  void *args[] = {&m, &p, &a};
  const uint32_t qw = query_waves(M), blocks = (A.n + qw - 1) / qw;
  hipError_t e = run_kernel(f, dim3(blocks < 8 * cus ? blocks : 8 * cus), kWave * qw, args, query_lds(M, qw), stream);
  if (e != hipSuccess) return e;
  e = run_kernel((const void *)fbs_layer_lists, dim3((A.n + kListPositions - 1) / kListPositions), 256, args, 4ull * M.D,
                 stream);
  if (e != hipSuccess) return e;
  const bool w32 = M.d % 64 == 0;
  f = w32 ? (t8 ? (const void *)fbs_layer_scan<32, true> : (const void *)fbs_layer_scan<32, false>)
          : (t8 ? (const void *)fbs_layer_scan<16, true> : (const void *)fbs_layer_scan<16, false>);
  ServeScan j = S;
  void *scan[] = {&m, &j};
  e = run_kernel(f, dim3(S.item_cap < 8 * cus ? S.item_cap : 8 * cus), kWave, scan, 0, stream);
  return e != hipSuccess ? e : launch_fbs_serve_finish(M, S, stream);
}

hipError_t launch_fbs_layer_choices(const LayerArgs &P, hipStream_t stream) {
  LayerArgs p = P;
  void *args[] = {&p};
  return run_kernel((const void *)fbs_layer_choices, dim3(P.n), 256, args, 0, stream);
}

}  // namespace fbs
