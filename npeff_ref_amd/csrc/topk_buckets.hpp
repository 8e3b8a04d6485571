// How top-k samples a row and deals the candidates to buckets: integer arithmetic that compiles for the host too.
#pragma once

#include <cmath>
#include <cstdint>

#if defined(__HIPCC__)
#define TOPK_HD __host__ __device__ inline
#else
#define TOPK_HD inline
#endif

namespace dn {

constexpr int TOPK_CHUNK = 64;            // sampled entries in a row
constexpr int TOPK_STRIDE = 2048;         // one chunk of every so many entries, or of twice as many
constexpr int64_t TOPK_SAMPLED = 1 << 19; // rows from this length on are sampled
constexpr int TOPK_MAX_LOG = 14;
constexpr int TOPK_MAX_BUCKETS = (1 << TOPK_MAX_LOG) + (1 << (TOPK_MAX_LOG - 2));
constexpr int TOPK_CROWDED = 2048;        // entries of a bucket that are still ranked one against the other

struct topk_plan {
  int64_t stride;   // a chunk of every so many entries is sampled
  unsigned target;  // entries of the sample to find above the threshold
  int64_t cap;      // room in the candidate list
  int log_nb, above;  // buckets: `above` for what is larger than all of the sample, 2^log_nb for the rest
  int buckets() const { return (1 << log_nb) + above; }
};
inline topk_plan topk_plan_of(int64_t count, int64_t k) {
  topk_plan p;
  const bool sampled = count >= TOPK_SAMPLED;
  p.stride = !sampled ? TOPK_CHUNK : k >= 8 * TOPK_STRIDE * 2 ? 2 * TOPK_STRIDE : TOPK_STRIDE;
  // entries of the sample to find above the threshold: their share of k and five times its deviation
  const double share = (double)k * TOPK_CHUNK / (double)p.stride;
  p.target = sampled ? (unsigned)(share + 5.0 * std::sqrt(share) + 8.0) : (unsigned)k;
  const double expected = sampled ? (double)p.target * p.stride / TOPK_CHUNK : (double)k;
  p.cap = (int64_t)(1.5 * expected) + 4096;
  if (p.cap > count) p.cap = count;
  p.log_nb = 8;
  while (p.log_nb < TOPK_MAX_LOG && ((int64_t)4 << p.log_nb) < p.cap) p.log_nb++;
  p.above = sampled ? 1 << (p.log_nb - 2) : 0;  // (sampled: log_nb is 11 at least)
  return p;
}

// Buckets of keys from the threshold up, the largest keys first: `above` buckets (0, or a power of two from 512 on) for
// keys past `top`, the largest sampled, then 2^log_nb buckets of 2^shift keys each from `top` down.  Past `top` a
// bucket's width grows with the distance, above / 32 buckets to every doubling of it: the few thousand entries that
// can lie between two chunks of the sample spread however far up they are.  In one bucket they send the row to the
// histograms of all entries: 20 M lognormal entries, 3072 larger ones in one gap, k = 65,536: 660 us, so 136.
// `top` is the largest key of the sample itself, not the end of its histogram bin, which spans a quarter of an
// octave: of 20 M entries 1 + 0.001 normal, k = 65,536, the fullest bucket has 84 (4286 with the bin's end, and the
// histograms again: 1130 us, so 140), of 20 M uniform in [0, 0.9) 16 (208; 171 us, so 127).
TOPK_HD int topk_shift(uint32_t thr, uint32_t top, int log_nb) {
  const uint32_t range = top - thr;
  const int bits = range ? 32 - __builtin_clz(range) : 0;
  return bits > log_nb ? bits - log_nb : 0;
}
TOPK_HD int topk_bucket(uint32_t key, uint32_t thr, uint32_t top, int shift, int above) {
  if (key <= top) return above + (int)(((top - thr) >> shift) - ((key - thr) >> shift));
  if (above == 0) return 0;  // (all entries are sampled: there is none)
  const uint32_t d = key - top;
  const int p = 31 - __builtin_clz(d), fine = 31 - __builtin_clz((unsigned)above) - 5;
  return above - 1 - (int)(((unsigned)p << fine) + ((d << (31 - p)) << 1 >> (32 - fine)));
}

}  // namespace dn

#undef TOPK_HD
