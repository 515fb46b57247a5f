// copy_read.hip - the copy heads' Hamming read on MI355X: for the last row of each token stream,
// every copy head picks earlier positions by the XOR-popcount distance between the row's query
// code and the positions' key codes under its rule, and the heads' margin-weighted mean of the
// table rows after those positions is the read (CopyHeads, crates/uor-r4-integer/src/stack/
// hamming.rs:266-538; nearest :690-701, latest_of :584-598, longest_of :601-615, mean_by
// :506-538).
//
// One wavefront reads one stream, four streams per block. The lanes take the candidate positions
// 64 at a time, four heads at once: under the mean rule the distances are staged in LDS with a
// histogram per head, whose running count gives the distance up to which positions are kept, and
// the kept ones are ranked by (distance, position); the latest and longest rules are wave minima
// and maxima over the matching positions. The weighted sums run with the lanes over the table
// row's coordinates, in 64-bit integers: a weight is at most 2^31 and a table value at most 2^15
// in magnitude, so a head's sum over at most 32 positions stays below 2^51.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/uor_copy.h"
#include "fbs_int.h"

namespace copyread {

constexpr int kWaves = 4;          // streams a block reads, one per wavefront
constexpr int kHeads = 4;          // heads that one pass over the positions serves
constexpr int kChunks = 4;         // chunks of 64 positions whose codes are in flight together
constexpr int kRows = 8;           // table rows in flight in a head's sum
constexpr uint32_t kBins = 68;     // distances 0..64, padded
constexpr uint32_t kPosBits = 20;  // positions below UOR_COPY_MAX_STRIDE fit
constexpr uint32_t kPosMask = (1u << kPosBits) - 1;
constexpr uint32_t kNone = 0xffffffffu;

struct Dev {
  uint32_t vocab, width, copy, kept, rule, has_marker, m0, m1;
  const uint64_t *codes;
  const int32_t *margins;
  const uint64_t *pair;
  const int16_t *table;
};

// A wavefront's LDS: the distances [kHeads][pitch] (bytes), the heads' histograms [kHeads][kBins],
// then one head's picked keys.
constexpr uint32_t kFixedLds = 4 * (kHeads * kBins + UOR_COPY_MAX_KEPT);
inline uint32_t wave_lds_bytes(uint32_t stride) { return kFixedLds + kHeads * ((stride + 63u) & ~63u); }

template <int CTRL>
__device__ __forceinline__ uint32_t dpp32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t lane32(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
// Wave minimum / maximum (DPP butterflies in each row of 16, then the rows as scalars).
__device__ __forceinline__ uint32_t wave_min32(uint32_t v) {
  v = min(v, dpp32<0xb1>(v));
  v = min(v, dpp32<0x4e>(v));
  v = min(v, dpp32<0x141>(v));
  v = min(v, dpp32<0x140>(v));
  return min(min(lane32(v, 0), lane32(v, 16)), min(lane32(v, 32), lane32(v, 48)));
}
__device__ __forceinline__ uint32_t wave_max32(uint32_t v) {
  v = max(v, dpp32<0xb1>(v));
  v = max(v, dpp32<0x4e>(v));
  v = max(v, dpp32<0x141>(v));
  v = max(v, dpp32<0x140>(v));
  return max(max(lane32(v, 0), lane32(v, 16)), max(lane32(v, 32), lane32(v, 48)));
}
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The value of the lane before, and `first` on lane 0.
__device__ __forceinline__ uint64_t lane_before(uint64_t v, uint64_t first) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)first, (int)(uint32_t)v, 0x138, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)(first >> 32), (int)(uint32_t)(v >> 32), 0x138, 0xf, 0xf, false);
  return (uint64_t)hi << 32 | lo;
}
__device__ __forceinline__ uint64_t lane64(uint64_t v, int l) {
  return (uint64_t)lane32((uint32_t)(v >> 32), l) << 32 | lane32((uint32_t)v, l);
}

__device__ __forceinline__ uint64_t code(const Dev &D, uint32_t token, uint32_t h) {
  return D.codes[(uint64_t)token * D.copy + h];
}
// The token's codes of heads h0 .. h0 + kHeads - 1 (a head past the last repeats the last): two
// 16-byte loads where the token's codes are whole pairs of them.
__device__ __forceinline__ void codes_of(const Dev &D, uint32_t token, uint32_t h0, uint64_t (&c)[kHeads]) {
  const uint64_t *at = D.codes + (uint64_t)token * D.copy;
  if (D.copy % kHeads == 0) {
    const ulonglong2 a = *(const ulonglong2 *)(at + h0), b = *(const ulonglong2 *)(at + h0 + 2);
    c[0] = a.x, c[1] = a.y, c[2] = b.x, c[3] = b.y;
  } else {
#pragma unroll
    for (int g = 0; g < kHeads; g++) c[g] = at[h0 + g < D.copy ? h0 + g : D.copy - 1];
  }
}
// joined (:379-385): under copy key 2 the near token's first half and the far token's second.
__device__ __forceinline__ uint64_t joined(uint64_t near, uint64_t far, uint64_t first) {
  return first ? (near & first) | (far & ~first) : near;
}

// floor(n / k) for n < 2^59 and k in [1, 32], without a division (the kernels divide by no
// variable with the compiler's `/`, whose expansion goes through a float reciprocal estimate): the
// high 64 bits of n m with m = ceil(2^64 / k), as m exceeds 2^64 / k by less than 1 and so n m / 2^64
// exceeds n / k by less than n / 2^64 < 1 / k.
struct Magic {
  uint64_t m[33];
};
constexpr Magic make_magic() {
  Magic g{};
  for (uint64_t k = 2; k <= 32; k++) g.m[k] = ~0ull / k + 1;  // m[1] stays 0: no factor below 2^64
  return g;
}
__constant__ const Magic kMagic = make_magic();
static_assert(UOR_COPY_MAX_KEPT <= 32 && UOR_COPY_MAX_HEADS <= 32, "the divisors' table");
// n / k rounded toward zero (Rust's i128 division): |n| is a sum of at most 32 products of 2^31
// and 2^15, or of 16 such quotients.
__device__ __forceinline__ int64_t div_trunc(int64_t n, uint64_t m) {
  const uint64_t q = m ? __umul64hi(fbs::uabs64(n), m) : fbs::uabs64(n);
  return n < 0 ? -(int64_t)q : (int64_t)q;
}

// copy_weight_q31 (:243-252), shared with the served step's reads.
__device__ __forceinline__ uint64_t weight_q31(int32_t margin, uint32_t d) {
  return fbs::copy_weight_q31(margin, d);
}

// One wavefront reads one stream. NV > 0: the lanes own four neighbouring coordinates each, NV
// groups of 256 (a width that is a multiple of 4, whose rows load as 8 bytes a lane); NV = 0:
// coordinates 64 apart, any width.
//
// Bound by latency: 4,096 streams are four wavefronts a SIMD, so the passes over the positions and
// the kept rows count by their round trips. One pass over the positions serves kHeads heads (a
// position's codes lie side by side) with the codes of kChunks chunks in flight, and the far key
// half comes from the lane before. Under the mean rule the distances go to LDS with a histogram
// a head; the kept positions are those below the distance at which the histogram reaches `kept`
// and the earliest at it, one further pass of ballots (the first form took `kept` successive wave
// minima, a pass each). The head's sum loads kRows rows at a time. 4,096 streams of up to 1,024
// tokens, 4 heads keeping 16: 505 us before, 94 us now.
template <int NV>
__global__ __launch_bounds__(64 * kWaves) void copy_mean_rows(Dev D, const uint32_t *__restrict__ tokens,
                                                              const int32_t *__restrict__ lengths,
                                                              const uint8_t *__restrict__ opening, uint32_t rows,
                                                              uint32_t stride, uint32_t pitch,
                                                              int64_t *__restrict__ out,
                                                              uint8_t *__restrict__ found,
                                                              int32_t *__restrict__ chosen) {
  constexpr int kVals = NV ? 4 * NV : UOR_COPY_MAX_WIDTH / 64;
  extern __shared__ __align__(16) uint8_t lds[];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint32_t row = blockIdx.x * (blockDim.x >> 6) + wave;
  if (row >= rows) return;
  uint8_t *mine = lds + wave * (kFixedLds + kHeads * pitch);
  uint32_t *hist = (uint32_t *)mine;
  uint32_t *pick = hist + kHeads * kBins;
  uint8_t *dist = mine + kFixedLds;
  const uint32_t *tok = tokens + (uint64_t)row * stride;
  int len = lengths[row];
  if (len < 0 || len > (int)stride) len = 0;  // outside the row: reads nothing
  const int t = len - 1;
  // The row's own token and the one before; a token outside the vocabulary reads nothing.
  const uint32_t raw_own = len ? tok[t] : 0, raw_prev = t > 0 ? tok[t - 1] : raw_own;
  bool bad = raw_own >= D.vocab || raw_prev >= D.vocab;
  const uint32_t own = bad ? 0 : raw_own, prev = bad ? 0 : raw_prev;
  const bool opens = D.has_marker ? (len >= 2 && raw_prev == D.m0 && raw_own == D.m1)
                                  : (opening != nullptr && opening[row] != 0);
  uint32_t rule = D.rule;
  if (rule == UOR_COPY_LONGEST_AFTER_OPENING)
    rule = opens ? UOR_COPY_LATEST_EXACT : UOR_COPY_LONGEST_EXACT;
  int64_t sum[kVals];
#pragma unroll
  for (int j = 0; j < kVals; j++) sum[j] = 0;
  int heads_found = 0;
  for (uint32_t h0 = 0; h0 < D.copy; h0 += kHeads) {
    uint64_t q[kHeads], first[kHeads], carry[kHeads], before[kHeads];
    {
      uint64_t a[kHeads], b[kHeads];
      codes_of(D, own, h0, a);
      codes_of(D, prev, h0, b);
#pragma unroll
      for (int g = 0; g < kHeads; g++) {
        first[g] = D.pair[h0 + g < D.copy ? h0 + g : D.copy - 1];
        q[g] = joined(a[g], b[g], first[g]);
        carry[g] = before[g] = 0;
      }
    }
    if (rule == UOR_COPY_LONGEST_EXACT && len && !bad) {
#pragma unroll
      for (int g = 0; g < kHeads; g++) {
        const int kd = first[g] ? 2 : 1;
        const uint32_t far = t >= kd ? tok[t - kd] : 0;
        before[g] = far < D.vocab ? code(D, far, h0 + g < D.copy ? h0 + g : D.copy - 1) : 0;
      }
    }
    for (uint32_t i = lane; i < kHeads * kBins; i += 64) hist[i] = 0;
    wave_sync();
    // Latest rules: least distance << 20 | (mask - s). Longest: the latest exact match and the
    // latest whose token before the key matches too.
    uint32_t best[kHeads], longer[kHeads];
#pragma unroll
    for (int g = 0; g < kHeads; g++) {
      best[g] = rule == UOR_COPY_LONGEST_EXACT ? 0 : kNone;
      longer[g] = 0;
    }
    for (int s0 = 1; s0 < t; s0 += 64 * kChunks) {
      uint32_t near[kChunks];
      uint64_t c[kChunks][kHeads];
#pragma unroll
      for (int u = 0; u < kChunks; u++) {
        const int s = s0 + 64 * u + (int)lane;
        near[u] = s < t ? tok[s - 1] : 0;
        bad |= near[u] >= D.vocab;
        near[u] = near[u] < D.vocab ? near[u] : 0;
      }
#pragma unroll
      for (int u = 0; u < kChunks; u++)
        if (s0 + 64 * u < t) codes_of(D, near[u], h0, c[u]);
#pragma unroll
      for (int u = 0; u < kChunks; u++) {
        if (s0 + 64 * u >= t) break;
        const int s = s0 + 64 * u + (int)lane;
        const bool in = s < t;
#pragma unroll
        for (int g = 0; g < kHeads; g++) {
          if (h0 + g >= D.copy) break;
          uint64_t far = 0;
          if (first[g]) {  // position 1's far token is its near one
            far = lane_before(c[u][g], s0 == 1 && u == 0 ? lane64(c[u][g], 0) : carry[g]);
            carry[g] = lane64(c[u][g], 63);
          }
          const uint32_t d = (uint32_t)__popcll(q[g] ^ joined(c[u][g], far, first[g]));
          if (rule == UOR_COPY_MEAN) {
            if (in) {
              dist[g * pitch + s] = (uint8_t)d;
              atomicAdd(&hist[g * kBins + d], 1u);
            }
          } else if (rule == UOR_COPY_LONGEST_EXACT) {
            if (in && d == 0) {
              const int kd = first[g] ? 2 : 1;
              best[g] = max(best[g], (uint32_t)s);
              const uint32_t past = s > kd ? tok[s - 1 - kd] : kNone;
              if (past < D.vocab && code(D, past, h0 + g) == before[g]) longer[g] = max(longer[g], (uint32_t)s);
            }
          } else if (in && (d == 0 || rule == UOR_COPY_LATEST_NEAREST)) {
            best[g] = min(best[g], d << kPosBits | (kPosMask - (uint32_t)s));
          }
        }
      }
    }
    bad = __any(bad);
    wave_sync();
#pragma unroll
    for (int g = 0; g < kHeads; g++) {
      const uint32_t h = h0 + g;
      if (h >= D.copy) break;
      // This head's picks, one a lane in the order read: (s | distance << 24); n of them.
      uint32_t mypick = 0;
      int n = 0;
      if (bad || t <= 1) {
        // nothing to read
      } else if (rule == UOR_COPY_MEAN) {
        // The distance `at` where the positions below it are fewer than `kept` and those up to it
        // are not (64 where the positions are no more than `kept`): lane b counts distance b.
        uint32_t upto = hist[g * kBins + lane];
        const uint32_t mineb = upto;
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
          const uint32_t o = (uint32_t)__shfl_up((int)upto, m, 64);
          upto += (int)lane >= m ? o : 0;
        }
        const uint64_t full = __ballot(upto >= D.kept);
        const uint32_t at = full ? (uint32_t)__ffsll((unsigned long long)full) - 1 : 64u;
        const uint32_t below = full ? lane32(upto - mineb, (int)at) : lane32(upto, 63);
        uint32_t lows = 0, ties = 0, tie_cap = D.kept - below;
        for (int s0 = 1; s0 < t; s0 += 64) {
          const int s = s0 + (int)lane;
          const uint32_t d = s < t ? dist[g * pitch + s] : 255u;
          const uint64_t lo = __ballot(d < at), eq = __ballot(d == at);
          if (lo | eq) {
            const uint64_t under = (1ull << lane) - 1;
            const uint32_t lr = lows + __popcll(lo & under), er = ties + __popcll(eq & under);
            if (d < at) pick[lr] = d << kPosBits | (uint32_t)s;
            if (d == at && er < tie_cap) pick[below + er] = d << kPosBits | (uint32_t)s;
            lows += __popcll(lo);
            ties += __popcll(eq);
          }
        }
        n = (int)(below + min(ties, tie_cap));
        wave_sync();
        // In (distance, position) order: a pick's place is the number of smaller keys.
        const uint32_t key = (int)lane < n ? pick[lane] : kNone;
        uint32_t place = 0;
        for (int k = 0; k < n; k++) place += lane32(key, k) < key ? 1u : 0u;
        wave_sync();
        if ((int)lane < n) pick[place] = (key & kPosMask) | (key >> kPosBits) << 24;
        wave_sync();
        mypick = (int)lane < n ? pick[lane] : 0;
      } else if (rule == UOR_COPY_LONGEST_EXACT) {
        const uint32_t ex = wave_max32(best[g]), lg = wave_max32(longer[g]);
        mypick = lg ? lg : ex;
        n = mypick != 0;
      } else {
        const uint32_t m = wave_min32(best[g]);
        if (m != kNone) {
          mypick = (kPosMask - (m & kPosMask)) | (m >> kPosBits) << 24;
          n = 1;
        }
      }
      if (chosen != nullptr && lane < D.kept)
        chosen[((uint64_t)row * D.copy + h) * D.kept + lane] = (int)lane < n ? (int32_t)mypick : -1;
      // Each pick's weight and row, a lane each. Weights fall with the distance, so those above
      // zero lead. The negated weight is at least -2^31, a signed 32-bit factor.
      const uint64_t wt = (int)lane < n ? weight_q31(D.margins[h], mypick >> 24) : 0;
      const uint32_t neg = 0u - (uint32_t)wt;
      const int count = __popcll(__ballot(wt != 0));
      if (count == 0) continue;
      const uint32_t rowtok = (int)lane < n ? tok[mypick & 0xffffff] : 0;
      int64_t head[kVals];
#pragma unroll
      for (int j = 0; j < kVals; j++) head[j] = 0;
      if constexpr (NV > 0) {
        for (int k0 = 0; k0 < count; k0 += kRows) {
          short4 v[kRows][NV];
#pragma unroll
          for (int k = 0; k < kRows; k++)
#pragma unroll
            for (int j = 0; j < NV; j++) {
              const uint32_t c = 4 * (lane + 64u * j);
              v[k][j] = make_short4(0, 0, 0, 0);
              if (k0 + k < count && c < D.width)
                v[k][j] = *(const short4 *)(D.table + (uint64_t)lane32(rowtok, k0 + k) * D.width + c);
            }
#pragma unroll
          for (int k = 0; k < kRows; k++) {
            const int32_t w = k0 + k < count ? (int32_t)lane32(neg, k0 + k) : 0;
#pragma unroll
            for (int j = 0; j < NV; j++) {
              head[4 * j] += (int64_t)v[k][j].x * w;
              head[4 * j + 1] += (int64_t)v[k][j].y * w;
              head[4 * j + 2] += (int64_t)v[k][j].z * w;
              head[4 * j + 3] += (int64_t)v[k][j].w * w;
            }
          }
        }
      } else {
        for (int k = 0; k < count; k++) {
          const int32_t w = (int32_t)lane32(neg, k);
          const int16_t *trow = D.table + (uint64_t)lane32(rowtok, k) * D.width;
#pragma unroll
          for (int j = 0; j < kVals; j++) {
            const uint32_t c = lane + 64u * j;
            if (c < D.width) head[j] += (int64_t)trow[c] * w;
          }
        }
      }
      heads_found++;
      const uint64_t m = kMagic.m[count];
#pragma unroll
      for (int j = 0; j < kVals; j++) sum[j] += div_trunc(-head[j], m);
    }
    wave_sync();
    if (bad) break;
  }
  if (bad) {  // every group of heads sees the same tokens, so the first one finds it
    heads_found = 0;
    if (chosen != nullptr)
      for (uint32_t i = lane; i < D.copy * D.kept; i += 64) chosen[(uint64_t)row * D.copy * D.kept + i] = -1;
  }
  const uint64_t m = kMagic.m[heads_found];
#pragma unroll
  for (int j = 0; j < kVals; j++) {
    const uint32_t c = NV ? 4 * (lane + 64u * (j / 4)) + j % 4 : lane + 64u * j;
    if (c < D.width) out[(uint64_t)row * D.width + c] = heads_found ? div_trunc(sum[j], m) : 0;
  }
  if (lane == 0) found[row] = heads_found > 0;
}

// vocab_codes (hamming.rs:566-582): one thread per (token, copy head); the sign word of the
// token's table point through the head's unit rotations (stack_hamilton, the unit on the left;
// the products are exact: |unit| <= 2^31, |point| <= 2^15).
__global__ void copy_vocab_codes(const int64_t *units, const int16_t *table, uint32_t vocab,
                                 uint32_t width, uint32_t head_width, uint32_t copy,
                                 uint64_t *codes) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (uint64_t)vocab * copy) return;
  const uint32_t v = (uint32_t)fbs::div128_64(i, copy), h = (uint32_t)(i - (uint64_t)v * copy);
  const int16_t *row = table + (uint64_t)v * width;
  uint64_t word = 0;
  for (uint32_t c = 0; c < head_width; c += 4) {
    const uint32_t at = h * head_width + c;
    const int64_t *a = units + at;  // the quaternion at / 4
    const int64_t b0 = row[at], b1 = row[at + 1], b2 = row[at + 2], b3 = row[at + 3];
    const int64_t r[4] = {a[0] * b0 - a[1] * b1 - a[2] * b2 - a[3] * b3,
                          a[0] * b1 + a[1] * b0 + a[2] * b3 - a[3] * b2,
                          a[0] * b2 - a[1] * b3 + a[2] * b0 + a[3] * b1,
                          a[0] * b3 + a[1] * b2 - a[2] * b1 + a[3] * b0};
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (r[k] >= 0) word |= 1ull << (c + k);
  }
  codes[i] = word;
}

thread_local std::string g_error;
int fail(int code, const std::string &m) {
  g_error = m;
  return code;
}

struct Handle {
  int device = 0;
  Dev d{};
  void *buf = nullptr;
  ~Handle() {
    int prev = 0;
    (void)hipGetDevice(&prev);
    (void)hipSetDevice(device);
    (void)hipFree(buf);
    (void)hipSetDevice(prev);
  }
};

}  // namespace copyread

using namespace copyread;

extern "C" uint32_t uor_copy_abi_version(void) { return UOR_COPY_ABI_VERSION; }
extern "C" const char *uor_copy_last_error(void) { return g_error.c_str(); }

extern "C" int uor_copy_create(const uor_copy_heads *m, int32_t device, void **handle) {
  if (!m || !handle) return fail(-1, "null argument");
  *handle = nullptr;
  if (m->vocabulary < 1 || m->width < 1 || m->width > UOR_COPY_MAX_WIDTH || m->copy < 1 ||
      m->copy > UOR_COPY_MAX_HEADS || m->kept < 1 || m->kept > UOR_COPY_MAX_KEPT ||
      m->rule > UOR_COPY_LONGEST_AFTER_OPENING)
    return fail(-1, "copy heads outside the supported shape");
  if (!m->codes || !m->margins_q16 || !m->pair_first || !m->table) return fail(-1, "null table");
  if (m->has_marker && (m->marker[0] >= m->vocabulary || m->marker[1] >= m->vocabulary))
    return fail(-1, "reply marker outside the vocabulary");
  const size_t nc = (size_t)m->vocabulary * m->copy * 8, nm = (size_t)m->copy * 4,
               np = (size_t)m->copy * 8, nt = (size_t)m->vocabulary * m->width * 2;
  const size_t oc = 0, om = (oc + nc + 255) & ~(size_t)255, op = (om + nm + 255) & ~(size_t)255,
               ot = (op + np + 255) & ~(size_t)255, total = ot + nt;
  int prev = 0;
  (void)hipGetDevice(&prev);
  if (hipSetDevice(device) != hipSuccess) return fail(-2, "hipSetDevice failed");
  Handle *h = new Handle();
  h->device = device;
  char *b = nullptr;
  bool ok = hipMalloc((void **)&b, total) == hipSuccess;
  if (ok) {
    h->buf = b;
    ok = hipMemcpy(b + oc, m->codes, nc, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b + om, m->margins_q16, nm, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b + op, m->pair_first, np, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(b + ot, m->table, nt, hipMemcpyHostToDevice) == hipSuccess;
  }
  (void)hipSetDevice(prev);
  if (!ok) {
    delete h;
    return fail(-2, "device allocation or copy failed");
  }
  h->d = Dev{m->vocabulary, m->width, m->copy, m->kept, m->rule, m->has_marker, m->marker[0],
             m->marker[1], (const uint64_t *)(b + oc), (const int32_t *)(b + om),
             (const uint64_t *)(b + op), (const int16_t *)(b + ot)};
  *handle = h;
  return 0;
}

extern "C" void uor_copy_destroy(void *handle) { delete (Handle *)handle; }

extern "C" int uor_copy_mean_rows_async(void *handle, const uint32_t *d_tokens,
                                        const int32_t *d_lengths, const uint8_t *d_opening,
                                        uint32_t rows, uint32_t stride, int64_t *d_out,
                                        uint8_t *d_found, int32_t *d_chosen, void *stream) {
  if (!handle) return fail(-1, "null handle");
  if (rows == 0) return 0;
  if (!d_tokens || !d_lengths || !d_out || !d_found || stride == 0 || stride > UOR_COPY_MAX_STRIDE)
    return fail(-1, "null buffer or stride outside 1..4096");
  Handle *h = (Handle *)handle;
  int prev = 0;
  (void)hipGetDevice(&prev);
  (void)hipSetDevice(h->device);
  // Four streams a block, or two where their distances would pass 64 KB of LDS (strides above
  // 3,776). The vector form wants rows of whole 8-byte pieces.
  const uint32_t pitch = (stride + 63u) & ~63u;
  const uint32_t waves = kWaves * wave_lds_bytes(stride) <= (64u << 10) ? kWaves : kWaves / 2;
  const uint32_t w = h->d.width;
  auto *kernel = w % 4 ? copy_mean_rows<0> : w <= 256 ? copy_mean_rows<1> : w <= 512 ? copy_mean_rows<2> : copy_mean_rows<4>;
  hipLaunchKernelGGL(kernel, dim3((rows + waves - 1) / waves), dim3(64 * waves), waves * wave_lds_bytes(stride),
                     (hipStream_t)stream, h->d, d_tokens, d_lengths, d_opening, rows, stride, pitch,
                     d_out, d_found, d_chosen);
  const hipError_t e = hipGetLastError();
  (void)hipSetDevice(prev);
  return e == hipSuccess ? 0 : fail(-2, std::string("launch: ") + hipGetErrorString(e));
}

extern "C" int uor_copy_mean_rows(void *handle, const uint32_t *tokens, const int32_t *lengths,
                                  const uint8_t *opening, uint32_t rows, uint32_t stride,
                                  int64_t *out, uint8_t *found, int32_t *chosen) {
  if (!handle) return fail(-1, "null handle");
  if (rows == 0) return 0;
  if (!tokens || !lengths || !out || !found || stride == 0 || stride > UOR_COPY_MAX_STRIDE)
    return fail(-1, "null buffer or stride outside 1..4096");
  Handle *h = (Handle *)handle;
  for (uint32_t r = 0; r < rows; r++) {
    if (lengths[r] < 0 || (uint32_t)lengths[r] > stride) return fail(-1, "a length exceeds the stride");
    for (int32_t i = 0; i < lengths[r]; i++)
      if (tokens[(size_t)r * stride + i] >= h->d.vocab) return fail(-1, "token outside the vocabulary");
  }
  const size_t nt = (size_t)rows * stride * 4, nl = (size_t)rows * 4, no = (size_t)rows * h->d.width * 8,
               nf = rows, nch = chosen ? (size_t)rows * h->d.copy * h->d.kept * 4 : 0;
  const size_t ot = 0, ol = (nt + 255) & ~(size_t)255, oo = (ol + nl + 255) & ~(size_t)255,
               of = (oo + no + 255) & ~(size_t)255, och = (of + nf + 255) & ~(size_t)255,
               oop = (och + nch + 255) & ~(size_t)255, total = oop + (opening ? rows : 0) + 16;
  int prev = 0;
  (void)hipGetDevice(&prev);
  (void)hipSetDevice(h->device);
  char *b = nullptr;
  int rc = 0;
  if (hipMalloc((void **)&b, total) != hipSuccess) {
    rc = fail(-2, "device allocation failed");
  } else {
    if (hipMemcpy(b + ot, tokens, nt, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b + ol, lengths, nl, hipMemcpyHostToDevice) != hipSuccess ||
        (opening && hipMemcpy(b + oop, opening, rows, hipMemcpyHostToDevice) != hipSuccess)) {
      rc = fail(-2, "copy to the device failed");
    } else {
      rc = uor_copy_mean_rows_async(handle, (const uint32_t *)(b + ot), (const int32_t *)(b + ol),
                                    opening ? (const uint8_t *)(b + oop) : nullptr, rows, stride,
                                    (int64_t *)(b + oo), (uint8_t *)(b + of),
                                    chosen ? (int32_t *)(b + och) : nullptr, nullptr);
      if (rc == 0 && (hipDeviceSynchronize() != hipSuccess ||
                      hipMemcpy(out, b + oo, no, hipMemcpyDeviceToHost) != hipSuccess ||
                      hipMemcpy(found, b + of, nf, hipMemcpyDeviceToHost) != hipSuccess ||
                      (chosen && hipMemcpy(chosen, b + och, nch, hipMemcpyDeviceToHost) != hipSuccess)))
        rc = fail(-2, "the read failed on the device");
    }
    (void)hipFree(b);
  }
  (void)hipSetDevice(prev);
  return rc;
}

extern "C" int uor_copy_vocab_codes(const int32_t *key_rotation, const int16_t *table,
                                    uint32_t vocab, uint32_t width, uint32_t heads_total,
                                    uint32_t copy, int32_t device, uint64_t *codes) {
  if (!key_rotation || !table || !codes) return fail(-1, "null buffer");
  if (vocab < 1 || width < 4 || width % 4 || heads_total < 1 || width % heads_total ||
      (width / heads_total) % 4 || width / heads_total > 64 || copy < 1 || copy > heads_total)
    return fail(-1, "codes need width / heads_total a multiple of 4 and at most 64");
  // The unit rotations g / |g| at Q31 (stack_rotation with lambda 2^31 and epsilon 0).
  std::vector<int64_t> units(width);
  for (uint32_t q = 0; q < width / 4; q++) fbs::rotation(key_rotation + 4 * q, 1ull << 31, 0, &units[4 * q]);
  const size_t nu = (size_t)width * 8, nt = (size_t)vocab * width * 2, nc = (size_t)vocab * copy * 8;
  const size_t ot = (nu + 255) & ~(size_t)255, oc = (ot + nt + 255) & ~(size_t)255;
  int prev = 0;
  (void)hipGetDevice(&prev);
  if (hipSetDevice(device) != hipSuccess) return fail(-2, "hipSetDevice failed");
  char *b = nullptr;
  int rc = 0;
  if (hipMalloc((void **)&b, oc + nc) != hipSuccess) {
    rc = fail(-2, "device allocation failed");
  } else {
    const uint64_t n = (uint64_t)vocab * copy;
    if (hipMemcpy(b, units.data(), nu, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b + ot, table, nt, hipMemcpyHostToDevice) != hipSuccess) {
      rc = fail(-2, "copy to the device failed");
    } else {
      hipLaunchKernelGGL(copy_vocab_codes, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, nullptr,
                         (const int64_t *)b, (const int16_t *)(b + ot), vocab, width,
                         width / heads_total, copy, (uint64_t *)(b + oc));
      if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
          hipMemcpy(codes, b + oc, nc, hipMemcpyDeviceToHost) != hipSuccess)
        rc = fail(-2, "the codes failed on the device");
    }
    (void)hipFree(b);
  }
  (void)hipSetDevice(prev);
  return rc;
}
