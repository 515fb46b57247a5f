// fbs_layers.hip - teacher-forced positions layer by layer: prompts taken in before a choice, and
// rows whose every position is scored.
//
// The step (RS stack/session.rs:4129-4403) runs one position after another because the next token
// is not known before the writer chose it. Where every token is known, only the recurrence's
// transport ties a position to the one before: a layer's norms, gathers, rotations, gates,
// requantizes and feed-forward block depend on the layer's input at that position alone, and the
// causal window on the drives of earlier positions. So these calls run each layer over all positions
// at once, in three kernels a layer: fbs_layer_front (a wavefront a position: the end of the layer
// before and the start of this one, up to the drives, the transitions and the output gates),
// fbs_layer_windows (a wavefront eight positions) and fbs_layer_chain (a lane a channel of a sequence:
// the state moved through the positions). A chain step is some 50 instructions against the step's 2,000
// a layer, so a prompt's time is set by the positions' work spread over the chip and no longer by the
// step's serial chain. The choices come from fbs_layer_query (final norm, Q12 query and drawer
// selection of each position) and the drawer-major scan of fbs_serve.hip, which reads a member row
// once for 16 positions.
// Every value is formed by the step's own routines (fbs_run.h), so the results are its bit for bit.
// At width 256 (window 16), 300 prompts of 509 tokens, microseconds a layer: front 450 (bound by its
// instructions, about 1,900 a position), windows 140, chain 225 (a serial 45 instructions a position).
#include "fbs_layers.h"
#include "fbs_run.h"

namespace fbs {

namespace {

constexpr uint32_t kFrontWaves = 4;  // wavefronts a block of fbs_layer_front, a position each
constexpr uint32_t kWindowWaves = 4;  // wavefronts a block of fbs_layer_windows
constexpr uint32_t kRun = 8;         // positions of each
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

// The end of layer l - 1 (the output gate on the moved state, rec_out, the feed-forward block; none
// at l = 0, where the position's table row comes in) and the start of layer l (none at l = L), for
// blockIdx.y's sequence, a wavefront a position.
template <int Q>
__global__ __launch_bounds__(64 * kFrontWaves, Q == 1 ? 3 : 2) void fbs_layer_front(DevModel M, LayerArgs P, uint32_t l) {
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
  // The layers' tables: held across the wavefront's positions, but loaded where they are used for four
  // quaternions a lane, whose registers would spill.
  constexpr bool kHold = Q < 4;
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
  if constexpr (kHold) load_out(), load_ffn(), load_down(), load_norm(), load_rec();
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
      if constexpr (!kHold) load_out();
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
      if constexpr (!kHold) load_ffn();
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
      if constexpr (!kHold) load_down();
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
      if constexpr (!kHold) load_norm();
      norm_publish<Q>(M, sd, x, qv, qi, g_rec, gd_rec, xbar);
      if constexpr (!kHold) load_rec();
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

// Layer l's windows (session.rs:4842-4868) for blockIdx.y's sequence, a wavefront 64 quaternions and
// kRun positions, into P.rhs. Tap k's word and row serve kRun positions: the rows of the positions lie
// in registers and move one place a tap, by naming and not by moving in each kRun taps.
__global__ __launch_bounds__(64 * kWindowWaves, 3) void fbs_layer_windows(DevModel M, LayerArgs P, uint32_t l) {
  const uint32_t lane = threadIdx.x % kWave, wave = uniform32(threadIdx.x / kWave);
  const uint32_t s = blockIdx.y, d = M.d, W = M.W, L = M.L;
  const uint32_t steps = P.steps[s];
  const uint32_t t0 = (blockIdx.x * kWindowWaves + wave) * kRun;
  const uint32_t q = blockIdx.z * kWave + lane;
  if (t0 >= steps || q >= M.nq) return;
  const uint32_t ch = 4 * q;
  const DevLayer ly = load_layer(M, l);
  const uint64_t p0 = (uint64_t)s * P.len;
  const int32_t *const drive = P.drive + p0 * d;
  const int32_t *const before = P.in_history ? P.in_history + ((uint64_t)s * L + l) * W * d : nullptr;
  const int32_t *const tw = M.tap_words + (uint64_t)l * (W + 1) * d;
  // The drive of position t (below t0 + kRun), or the session's row -1 - t; none before them (the terms
  // of a zero row are 0), nor past the last position.
  const auto row = [&](int32_t t) {
    if (t >= 0) return (uint32_t)t < steps ? gat<int4>(drive, 4 * ((uint32_t)t * d + ch)) : make_int4(0, 0, 0, 0);
    return before && t >= -(int32_t)W ? gat<int4>(before, 4 * ((uint32_t)(-1 - t) * d + ch)) : make_int4(0, 0, 0, 0);
  };
  const int4 bias = gat<int4>(ly.conv_bias, 4 * ch);
  int64_t acc[kRun][4];
  int4 rows[kRun];  // at tap k, position t0 + u's row t0 + u - k is rows[(u - k) mod kRun]
#pragma unroll
  for (uint32_t u = 0; u < kRun; u++) {
    acc[u][0] = bias.x, acc[u][1] = bias.y, acc[u][2] = bias.z, acc[u][3] = bias.w;
    rows[u] = row((int32_t)(t0 + u));
  }
#pragma unroll 1
  for (uint32_t k0 = 0; k0 <= W; k0 += kRun) {
    int4 tap[kRun], next[kRun];
#pragma unroll
    for (uint32_t j = 0; j < kRun; j++) {
      const uint32_t k = k0 + j;
      if (k <= W) tap[j] = gat<int4>(tw, 4 * (k * d + ch));
      if (k < W) next[j] = row((int32_t)t0 - 1 - (int32_t)k);
    }
#pragma unroll
    for (uint32_t j = 0; j < kRun; j++) {
      if (k0 + j > W) break;
#pragma unroll
      for (uint32_t u = 0; u < kRun; u++) add_tap(rows[(u + kRun - j) % kRun], tap[j], acc[u]);
      // The last position's row leaves, the one before the first's enters in its place.
      rows[kRun - 1 - j] = next[j];
    }
  }
#pragma unroll
  for (uint32_t u = 0; u < kRun; u++)
    if (t0 + u < steps) {
      longlong2 *o = (longlong2 *)(P.rhs + (p0 + t0 + u) * d + ch);
      o[0] = make_longlong2(acc[u][0], acc[u][1]);
      o[1] = make_longlong2(acc[u][2], acc[u][3]);
    }
}

// The value of another lane of the lane's quad (quad_perm CTRL).
template <int CTRL>
__device__ __forceinline__ int32_t quad(uint32_t v) {
  return __builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}

// Layer l's transport (session.rs:5097-5145) for blockIdx.y's sequence, a lane a channel: the window
// sums in P.rhs give way to the moved state at the residual's exponent. The four lanes of a
// quaternion exchange its halves by DPP: component k of T (x) b is the sum over i of +-T_i b_(k xor i),
// so a lane makes four products of each half and not the sixteen of a whole quaternion. The state of
// kAhead positions moves by transport_fast's form without a branch; where one left its ranges, they
// move again from the state before them in 128 bits. Lanes past the width repeat the last quaternion.
__global__ __launch_bounds__(64, 2) void fbs_layer_chain(DevModel M, LayerArgs P, uint32_t l) {
  constexpr uint32_t kAhead = 8;
  const uint32_t lane = threadIdx.x, k = lane % 4;
  const uint32_t s = blockIdx.y, d = M.d, nq = M.nq, L = M.L, W = M.W;
  const uint32_t c0 = blockIdx.x * kWave + lane, ch = c0 < d ? c0 : d - 4 + k;
  const uint32_t steps = P.steps[s];
  const uint64_t p0 = (uint64_t)s * P.len;
  const int32_t *const turn = P.turn + p0 * d;
  const uint32_t *const keeps = P.keep + p0 * nq;
  int64_t *const sums = P.rhs + p0 * d;
  // The signs of T_1..T_3 in component k: masks and their negations.
  const int32_t s1 = k == 0 || k == 2 ? -1 : 0, s2 = k == 0 || k == 3 ? -1 : 0, s3 = k < 2 ? -1 : 0;
  const int32_t n1 = -s1, n2 = -s2, n3 = -s3;
  int64_t h = P.in_state ? P.in_state[((uint64_t)s * L + l) * d + ch] : 0;
  struct Ops {
    int4 T;
    int64_t wide;
    uint32_t keep;
  };
  const auto fetch = [&](uint32_t t0, Ops (&o)[kAhead]) {
#pragma unroll
    for (uint32_t i = 0; i < kAhead; i++) {
      const uint32_t t = t0 + i < steps ? t0 + i : steps - 1;
      o[i].T = gat<int4>(turn + (uint64_t)t * d, 4 * (ch & ~3u));
      o[i].wide = gat<int64_t>(sums + (uint64_t)t * d, 8 * ch);
      o[i].keep = gat<uint32_t>(keeps + (uint64_t)t * nq, ch & ~3u);
    }
  };
  const auto store = [&](uint32_t t, int64_t rhs) { sums[(uint64_t)t * d + ch] = rhs; };
  const auto move = [&](uint32_t t0, const Ops (&o)[kAhead]) {
    const uint32_t n = steps - t0 < kAhead ? steps - t0 : kAhead;
    const int64_t h0 = h;
    uint32_t out_h = 0, out_w = 0;  // bits 28.. and 14..: a product or a window sum past transport_fast's ranges
    if (__all(split_ok(h))) {
      int64_t rhs[kAhead];
#pragma unroll
      for (uint32_t i = 0; i < kAhead; i++) {
        if (i >= n) continue;
        const int4 T = o[i].T;
        const int32_t a1 = (T.y ^ s1) + n1, a2 = (T.z ^ s2) + n2, a3 = (T.w ^ s3) + n3;
        const uint32_t hi = (uint32_t)(((uint64_t)h + (1ull << 31)) >> 32), lo = (uint32_t)h;
        const int32_t wh = (int32_t)(o[i].wide >> 32), keep = (int32_t)o[i].keep;
        const uint64_t K = (uint64_t)o[i].keep * (uint32_t)o[i].wide;
        uint32_t z0 = (((uint32_t)K & 0x7fffu) << 16) + (1u << 30);
        asm("" : "+v"(z0));  // added as 32 bits, not again as 64
        const int64_t H = (int64_t)T.x * (int32_t)hi + (int64_t)a1 * quad<0xB1>(hi) + (int64_t)a2 * quad<0x4E>(hi) +
                          (int64_t)a3 * quad<0x1B>(hi);
        const int64_t Z = (int64_t)(uint64_t)z0 + (int64_t)T.x * (int32_t)lo + (int64_t)a1 * quad<0xB1>(lo) +
                          (int64_t)a2 * quad<0x4E>(lo) + (int64_t)a3 * quad<0x1B>(lo);
        out_h |= (uint32_t)(H >> 32) + (1u << 27);
        out_w |= (uint32_t)wh + (1u << 13);
        // transport_fast(H, L, keep, wide)
        h = (int64_t)(((uint64_t)(H + (int64_t)keep * (int32_t)((uint32_t)wh << 16)) << 1) + (K >> 15)) + (Z >> 31);
        rhs[i] = (h + (1ll << 15)) >> 16;  // |h| < 2^62: the sum does not saturate
      }
      if (!__any((out_h >> 28) | (out_w >> 14))) {
#pragma unroll
        for (uint32_t i = 0; i < kAhead; i++)
          if (i < n) store(t0 + i, rhs[i]);
        return;
      }
    }
    h = h0;
#pragma unroll 1
    for (uint32_t t = t0; t < t0 + n; t++) {
      const int4 T = gat<int4>(turn + (uint64_t)t * d, 4 * (ch & ~3u));
      const int64_t wide = gat<int64_t>(sums + (uint64_t)t * d, 8 * ch);
      const uint32_t keep = gat<uint32_t>(keeps + (uint64_t)t * nq, ch & ~3u);
      const uint64_t v = (uint64_t)h;
      const int32_t a[4] = {T.x, T.y, T.z, T.w};
      const int64_t b[4] = {(int64_t)dpp64<0x00>(v), (int64_t)dpp64<0x55>(v), (int64_t)dpp64<0xAA>(v),
                            (int64_t)dpp64<0xFF>(v)};
      int64_t H[4], Lo[4];
      hamilton32_hl(a, b, H, Lo);
      const int64_t hk = k == 0 ? H[0] : k == 1 ? H[1] : k == 2 ? H[2] : H[3];
      const int64_t lk = k == 0 ? Lo[0] : k == 1 ? Lo[1] : k == 2 ? Lo[2] : Lo[3];
      const u128 term = (u128)((i128)(uint64_t)keep * (i128)wide) << 16;  // as transport_wide
      h = shift_wide((i128)((u128)(((i128)hk << 32) + (i128)lk) + term), 31);
      store(t, shift(h, kResidualExp - kStateExp));
    }
  };
  if (steps) {
    Ops a[kAhead], b[kAhead];
    fetch(0, a);
    for (uint32_t t = 0; t < steps; t += 2 * kAhead) {
      if (t + kAhead < steps) fetch(t + kAhead, b);
      move(t, a);
      if (t + 2 * kAhead < steps) fetch(t + 2 * kAhead, a);
      if (t + kAhead < steps) move(t + kAhead, b);
    }
  }
  if (steps < P.len || !P.out_state) return;  // a refused sequence exports nothing
  P.out_state[((uint64_t)s * L + l) * d + ch] = h;
  // Row r is the drive r + 1 positions back; the oldest first, so that the rows may be the ones that
  // came in.
  const int32_t *const drive = P.drive + p0 * d + ch;
  const int32_t *const before = P.in_history ? P.in_history + ((uint64_t)s * L + l) * W * d + ch : nullptr;
  int32_t *const out = P.out_history + ((uint64_t)s * L + l) * W * d + ch;
  for (int32_t r = (int32_t)W - 1; r >= 0; r--) {
    int32_t v = 0;
    if ((uint32_t)r < P.len)
      v = drive[(uint64_t)(P.len - 1 - r) * d];
    else if (before)
      v = before[(uint64_t)(r - P.len) * d];
    out[(uint64_t)r * d] = v;
  }
}

// The final norm, the Q12 query and the drawer selection of A.n positions from P.first on, a wavefront
// each; each position's job for the drawer-major scan.
template <int Q, bool T8>
__global__ __launch_bounds__(64) void fbs_layer_query(DevModel M, LayerArgs P, RunArgs A) {
  extern __shared__ __align__(16) int32_t lds[];
  const uint32_t lane = threadIdx.x, i = blockIdx.x, d = M.d;
  const uint32_t p = P.first + i;
  uint32_t s = (uint32_t)((p * P.len_recip) >> 32);  // p / len, or one less
  uint32_t t = p - s * P.len;
  if (t >= P.len) s++, t -= P.len;
  if (t >= P.steps[s] || (!P.out_tokens && P.start + t + 1 == P.row)) return;
  const uint64_t at_row = (uint64_t)s * P.row + P.start + t;  // its place in the rows
  uint32_t *seeds = (uint32_t *)lds;
  for (uint32_t k = lane; k < kSeedWords; k += kWave)
    seeds[k] = k < kRsqrtSeedWords ? rsqrt_seed_table()[k] : recip_seed_table()[k - kRsqrtSeedWords];
  const Seeds sd(seeds, seeds + kRsqrtSeedWords);
  int32_t *query = lds + kSeedWords;
  uint32_t *kept = (uint32_t *)(query + d), *dscore = kept + kMaxProbes;
  wave_sync();
  bool qv[Q];
  uint32_t qi[Q];
  int32_t x[Q][4];
  short4 g[Q];
  uint2 gd[Q];
#pragma unroll
  for (int k = 0; k < Q; k++) {
    qi[k] = lane + kWave * k;
    qv[k] = qi[k] < M.nq;
    const uint32_t at = 4 * (qv[k] ? qi[k] : 0);
    int4 v = *(const int4 *)(P.x + (uint64_t)p * d + at);
    if (!qv[k]) v = make_int4(0, 0, 0, 0);
    x[k][0] = v.x, x[k][1] = v.y, x[k][2] = v.z, x[k][3] = v.w;
    g[k] = *(const short4 *)(M.final_gain + at);
    gd[k] = *(const uint2 *)(M.final_gain_desc + at);
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
  if (P.out_kept && lane < M.P) P.out_kept[at_row * M.P + lane] = kept[lane];
  push_job<Q, T8>(M, A, i, query, kept, lane, qv, qi);
}

// The stretch's choices to the rows' place and their matches with the rows' next tokens.
__global__ __launch_bounds__(256) void fbs_layer_choices(LayerArgs P) {
  const uint32_t s = blockIdx.x;
  const uint32_t steps = P.steps[s];
  const uint32_t *tok = P.tokens + (uint64_t)s * P.row + P.start;
  uint32_t hits = 0;
  for (uint32_t t = threadIdx.x; t < steps; t += blockDim.x) {
    const bool next = P.start + t + 1 < P.row;
    if (!P.out_tokens && !next) continue;
    const uint32_t c = P.chosen[(uint64_t)s * P.len + t];
    if (P.out_tokens) P.out_tokens[(uint64_t)s * P.row + P.start + t] = c;
    hits += next && c == tok[t + 1];
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
size_t query_lds(const DevModel &M) { return 4ull * (kSeedWords + M.d + kMaxProbes + ((M.D + 3u) & ~3u)); }

// The front kernel's wavefronts a block: four, or fewer where wide layers' crossbars need the room.
uint32_t front_waves(const DevModel &M) {
  for (uint32_t w = kFrontWaves; w > 0; w /= 2)
    if (front_lds(M, w) <= kLayerLds) return w;
  return 0;
}
}  // namespace

bool fbs_layers_fit(const DevModel &M) {
  return front_waves(M) != 0 && query_lds(M) <= kLayerLds;
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
  const uint32_t waves = front_waves(M), per = waves * P.turns, win = kWindowWaves * kRun;
  for (l = 0; l < M.L + (rows ? 1u : 0u) && e == hipSuccess; l++) {
    e = run_kernel(front, dim3((P.len + per - 1) / per, P.n), kWave * waves, args, front_lds(M, waves), stream);
    if (l == M.L) break;
    if (e == hipSuccess)
      e = run_kernel((const void *)fbs_layer_windows, dim3((P.len + win - 1) / win, P.n, (M.nq + kWave - 1) / kWave),
                     kWave * kWindowWaves, args, 0, stream);
    if (e == hipSuccess)
      e = run_kernel((const void *)fbs_layer_chain, dim3((M.d + kWave - 1) / kWave, P.n), kWave, args, 0, stream);
  }
  return e;
}

hipError_t launch_fbs_layer_query(const DevModel &M, const LayerArgs &P, const RunArgs &A, hipStream_t stream) {
  DevModel m = M;
  LayerArgs p = P;
  RunArgs a = A;
  void *args[] = {&m, &p, &a};
  const bool t8 = M.table8 != nullptr;
  const void *f = M.qpl == 1 ? (t8 ? (const void *)fbs_layer_query<1, true> : (const void *)fbs_layer_query<1, false>)
                  : M.qpl == 2
                      ? (t8 ? (const void *)fbs_layer_query<2, true> : (const void *)fbs_layer_query<2, false>)
                      : (t8 ? (const void *)fbs_layer_query<4, true> : (const void *)fbs_layer_query<4, false>);
  return run_kernel(f, dim3(A.n), kWave, args, query_lds(M), stream);
}

hipError_t launch_fbs_layer_choices(const LayerArgs &P, hipStream_t stream) {
  LayerArgs p = P;
  void *args[] = {&p};
  return run_kernel((const void *)fbs_layer_choices, dim3(P.n), 256, args, 0, stream);
}

}  // namespace fbs
