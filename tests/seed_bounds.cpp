// Exhaustive checks of the kernels' reciprocal and reciprocal-square-root estimates
// (uor-r4_amd/csrc/fbs_int.h), over every input they take:
//   rsqrt_q46(t), t in [2^30, 2^32): within 2^-28.9 of 2^46 / sqrt(t), in [2^30, 2^31], and equal
//     to the same Newton iteration carried in 64-bit products;
//   rsqrt_q46s(t), the same t: within 2^-28.3 of 2^46 / sqrt(t), below 2^31;
//   rsqrt_q86(xn), xn = t 2^32 + b for every t, at b = 0 and 2^32 - 1 and, for every eighth t, one b
//     between (its error depends on b only by the products' floors): within (-2, +0.1] of
//     2^86 / sqrt(xn), in [2^54 - 1, 2^55];
//   recip_q63(d), d in [2^31, 2^32): within [-2^-30.4, 0] of 2^63 / d, below 2^32, and equal to the
//     same iteration in 64-bit products.
// The comparisons of error use long double (a test, not served code). Prints one line per routine
// with its mismatch count and worst errors; exits nonzero on any failure.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <thread>
#include <vector>

#include "../uor-r4_amd/csrc/fbs_int.h"

using namespace fbs;

static uint32_t rsqrt_wide(uint32_t t, const uint32_t *tab) {
  uint64_t y = tab[(t >> 23) - 128];
  for (int it = 0; it < 2; it++) {
    uint64_t y2 = (y * y) >> 32, p = ((uint64_t)t * y2) >> 28, f = ((3ull << 32) - p) >> 1;
    y = (y * f) >> 32;
    if (y > (1ull << 31)) y = 1ull << 31;
    if (y < (1ull << 30)) y = 1ull << 30;
  }
  return (uint32_t)y;
}
static uint64_t recip_wide(uint32_t d, const uint32_t *tab) {
  uint64_t w = tab[(d >> 23) - 256];
  for (int it = 0; it < 2; it++) {
    int64_t e = (int64_t)((1ull << 63) - (uint64_t)d * w);
    w = (uint64_t)((int64_t)w + (((e >> 31) * (int64_t)w) >> 32));
  }
  return w;
}

struct Acc {
  uint64_t bad = 0;
  long double lo = 0, hi = 0;
};

// 2^-28.9, 2^-28.3 and 2^-30.4.
static const long double kRsqrt = std::pow(2.0L, -28.9L), kRsqrtS = std::pow(2.0L, -28.3L),
                         kRecip = std::pow(2.0L, -30.4L);

int main() {
  const unsigned T = std::thread::hardware_concurrency() ? std::thread::hardware_concurrency() : 4;
  const uint32_t *rt = rsqrt_seed_table(), *ct = recip_seed_table();
  std::vector<Acc> ra(T), sa(T), qa(T), ca(T);
  std::vector<std::thread> th;
  for (unsigned k = 0; k < T; k++)
    th.emplace_back([&, k] {
      Acc a, b, q, c;  // the thread's own, not beside another's
      const uint64_t lo = 1ull << 30, n = 3ull << 30;
      const uint64_t begin = lo + k * (n / T), end = lo + (k + 1 == T ? n : (k + 1) * (n / T));
      const auto root = [](uint64_t t) { return 0x1p46L / std::sqrt((long double)t); };
      long double exact = root(begin);
      for (uint64_t t = begin; t < end; t++) {
        const long double after = root(t + 1);
        const uint32_t y = rsqrt_q46((uint32_t)t, rt);
        const long double rel = ((long double)y - exact) / exact;
        a.lo = rel < a.lo ? rel : a.lo;
        a.hi = rel > a.hi ? rel : a.hi;
        a.bad += y != rsqrt_wide((uint32_t)t, rt) || y < (1u << 30) || y > (1u << 31) ||
                 std::fabs(rel) > kRsqrt;
        const uint32_t z = rsqrt_q46s((uint32_t)t, rt);
        const long double srel = ((long double)z - exact) / exact;
        b.lo = srel < b.lo ? srel : b.lo;
        b.hi = srel > b.hi ? srel : b.hi;
        b.bad += z >= (1u << 31) || std::fabs(srel) > kRsqrtS;
        // 2^86 / sqrt(t 2^32 + b) is 2^24 times the root between those of t and t + 1, which it follows
        // along a straight line (its bend over one t is below 2^-7 of the result's units).
        const uint32_t lows[] = {0u, 0xffffffffu, (uint32_t)t * 2654435761u};
        for (int i = 0; i < (t % 8 ? 2 : 3); i++) {
          const uint32_t low = lows[i];
          const uint64_t r = rsqrt_q86(t << 32 | low, rt);
          const long double want = 0x1p24L * exact + (after - exact) * (0x1p-8L * low);
          const long double err = (long double)r - want;
          q.lo = err < q.lo ? err : q.lo;
          q.hi = err > q.hi ? err : q.hi;
          q.bad += err <= -2.0L || err > 0.1L || r < (1ull << 54) - 1 || r > (1ull << 55);
        }
        exact = after;
      }
      const uint64_t dlo = 1ull << 31, dn = 1ull << 31;
      for (uint64_t d = dlo + k * (dn / T); d < dlo + (k + 1 == T ? dn : (k + 1) * (dn / T)); d++) {
        const uint64_t w = recip_q63((uint32_t)d, ct);
        const long double exact = 0x1p63L / (long double)d;
        const long double rel = ((long double)w - exact) / exact;
        c.lo = rel < c.lo ? rel : c.lo;
        c.hi = rel > c.hi ? rel : c.hi;
        c.bad += w != recip_wide((uint32_t)d, ct) || w >= (1ull << 32) ||
                 rel < -kRecip || rel > 0;
      }
      ra[k] = a, sa[k] = b, qa[k] = q, ca[k] = c;
    });
  for (auto &t : th) t.join();
  const auto merge = [T](const std::vector<Acc> &from) {
    Acc r;
    for (unsigned k = 0; k < T; k++) {
      r.bad += from[k].bad;
      r.lo = from[k].lo < r.lo ? from[k].lo : r.lo, r.hi = from[k].hi > r.hi ? from[k].hi : r.hi;
    }
    return r;
  };
  const Acc r = merge(ra), s = merge(sa), q = merge(qa), c = merge(ca);
  printf("rsqrt_q46 bad %llu rel [%.3Lf, %.3Lf] (log2 |.|)\n", (unsigned long long)r.bad,
         r.lo ? std::log2(-r.lo) : -99.0L, r.hi ? std::log2(r.hi) : -99.0L);
  printf("rsqrt_q46s bad %llu rel [%.3Lf, %.3Lf] (log2 |.|)\n", (unsigned long long)s.bad,
         s.lo ? std::log2(-s.lo) : -99.0L, s.hi ? std::log2(s.hi) : -99.0L);
  printf("rsqrt_q86 bad %llu error [%.3Lf, %.3Lf]\n", (unsigned long long)q.bad, q.lo, q.hi);
  printf("recip_q63 bad %llu rel [%.3Lf, %.3Lf] (log2 |.|)\n", (unsigned long long)c.bad,
         c.lo ? std::log2(-c.lo) : -99.0L, c.hi ? std::log2(c.hi) : -99.0L);
  return r.bad || s.bad || q.bad || c.bad;
}
