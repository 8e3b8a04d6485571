// Per-example top-k of dense Fisher rows on the device: the sparsifier that produces the PEF
// rows the loader reads (values and indices of the k largest entries in descending order, equal
// values in ascending index order, plus the L2 norm of the whole row), i.e. what
// npeff/fishers/d_pefs_computer.py:126-129 gets from tf.math.top_k and :48-50 from the einsum.
//
// A row has ~1e8 entries and k ~ 6.5e4, so sorting the row is out of the question.  Usual case, one read
// of the row and a thirty-second of it before:
//   1. two histograms (11 bits of an order-preserving integer key each) of a sample, 64 entries out
//      of every 2048 (of every 4096, half the lines, where k leaves 512 of them above the threshold), give a threshold that a little more than k entries reach (all entries
//      of a short row: exactly the k-th entry's 22 bits);
//   2. every entry from the threshold up goes to a candidate list ((key, index) pairs, any order) and is
//      counted into its bucket (topk_buckets.hpp), and the sum of squares is taken on the way;
//   3. the candidates are placed into their buckets by the count that they met (an atomic of their own on a
//      cursor each took 18 us at 2 x 72,000 candidates, now 5; counting them after the collection 14 more); an
//      entry's place is its bucket's start plus the number of larger pairs in the bucket.
// When the threshold was too high (fewer than k candidates), when far more entries reach it than
// expected, or when a bucket is crowded (many equal entries), the row goes through histograms of all
// entries instead: 11 bits find the bin of the k-th entry, that bin and all above it are sorted
// (bitonic, strides below 4096 inside LDS); if the bin is crowded, one or two more histogram passes (11
// + 10 bits) narrow it down first; if even the entries equal to the exact key T of the k-th entry are
// too many to sort, the entries above T and the first `need` entries equal to T in index order (a
// predicate scan) are the candidates.  Everything but the norm is integer work; nothing depends on
// scheduling.
#include "dnpeff_internal.hpp"
#include "host_parts.hpp"
#include "scan.hpp"
#include "topk_buckets.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

namespace dn {

// Order-preserving key of a float: larger float <=> larger unsigned key (NaNs sort above +inf).
__device__ inline uint32_t sort_key(float x) {
  const uint32_t b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ inline float key_to_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

struct TopkState {
  uint32_t prefix;  // bits of T decided so far
  uint32_t mask;    // which bits those are
  int64_t need;     // entries still to take among those matching the prefix
  int64_t cursor;   // next free candidate slot (compaction)
  int64_t in_bin;   // entries in the bin picked last
};

constexpr int TOPK_BINS = 2048;

__global__ void __launch_bounds__(256) k_topk_init(TopkState* st, int64_t k) {
  st[blockIdx.x] = TopkState{0u, 0u, k, 0, 0};
}

// hist[row][bin] += entries of the row whose decided bits match and whose next `bits` bits are bin
template <bool VEC4>
__global__ void __launch_bounds__(256)
    k_topk_hist(const float* __restrict__ x, int64_t count, int shift, int bits,
                const TopkState* __restrict__ st, unsigned* __restrict__ hist,
                double* __restrict__ sq_partials) {
  __shared__ unsigned h[TOPK_BINS];
  __shared__ double red[256];
  double sq = 0.0;
  const int row = blockIdx.y;
  const uint32_t prefix = st[row].prefix, mask = st[row].mask;
  const unsigned nb = 1u << bits;
  for (unsigned i = threadIdx.x; i < nb; i += 256) h[i] = 0;
  __syncthreads();
  const float* xr = x + (int64_t)row * count;
  const int64_t stride = (int64_t)gridDim.x * 256;
  auto one = [&](float v) {
    const uint32_t key = sort_key(v);
    if ((key & mask) == prefix) atomicAdd(&h[(key >> shift) & (nb - 1)], 1u);
    sq += (double)v * (double)v;
  };
  if (VEC4) {  // count % 4 == 0 and x 16-byte aligned: four entries per load
    const float4* x4 = reinterpret_cast<const float4*>(xr);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count / 4; i += stride) {
      const float4 v = x4[i];
      one(v.x); one(v.y); one(v.z); one(v.w);
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += stride) one(xr[i]);
  }
  __syncthreads();
  for (unsigned i = threadIdx.x; i < nb; i += 256)
    if (h[i]) atomicAdd(&hist[(int64_t)row * TOPK_BINS + i], h[i]);
  if (sq_partials) {  // fixed tree inside the block, blocks summed in order by k_topk_norm
    red[threadIdx.x] = sq;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
      if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
      __syncthreads();
    }
    if (threadIdx.x == 0) sq_partials[(int64_t)row * gridDim.x + blockIdx.x] = red[0];
  }
}

__global__ void __launch_bounds__(64)
    k_topk_norm(const double* __restrict__ sq_partials, int n_partials, float* __restrict__ norms) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n_partials; i += 64) s += sq_partials[(int64_t)blockIdx.x * n_partials + i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (threadIdx.x == 0) norms[blockIdx.x] = (float)sqrt(s);
}

// Walks the bins from the top until `need` entries are covered; fixes the next bits of T.
__global__ void __launch_bounds__(64)
    k_topk_pick(unsigned* __restrict__ hist, int shift, int bits, TopkState* __restrict__ st) {
  const int row = blockIdx.x;
  unsigned* h = hist + (int64_t)row * TOPK_BINS;
  if (threadIdx.x == 0) {
    TopkState s = st[row];
    const int nb = 1 << bits;
    int64_t above = 0;
    int b = nb - 1;
    for (; b > 0; b--) {
      if (above + h[b] >= s.need) break;
      above += h[b];
    }
    s.prefix |= (uint32_t)b << shift;
    s.mask |= (uint32_t)(nb - 1) << shift;
    s.need -= above;
    s.in_bin = h[b];
    st[row] = s;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < TOPK_BINS; i += 64) h[i] = 0;
}

// A wave's finds on their way to a row's candidate list.  They wait in LDS and room in the list is reserved
// once per 256+ of them: the finds are sparse (k of ~1e8), and one global atomic each on a single counter
// would serialise them.  Every wave keeps its own buffer and count, so the loop that reads the row has no
// barrier in it.
struct topk_finds {
  uint64_t* buf;  // 512 slots
  unsigned n;     // the same in every lane
  uint64_t* out;
  int64_t cap;
  unsigned long long* cursor;
  int* buckets;  // (or NULL) entries per bucket, counted as they are written: `place` receives the count before
  unsigned* place;
  uint32_t thr, top;
  int shift, above;

  // All lanes call these together.
  __device__ void put(bool take, uint32_t key, int64_t i) {
    const uint64_t who = __ballot(take);
    const unsigned before = __builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0u));
    if (take) buf[n + before] = ((uint64_t)key << 32) | (uint32_t)(0xffffffffu - (uint32_t)i);
    n += (unsigned)__popcll(who);
  }
  __device__ void write(unsigned long long base) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (unsigned i = threadIdx.x & 63; i < n; i += 64)
      if (base + i < (unsigned long long)cap) {
        out[base + i] = buf[i];
        if (buckets) place[base + i] = (unsigned)atomicAdd(&buckets[topk_bucket((uint32_t)(buf[i] >> 32), thr, top, shift, above)], 1);
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    n = 0;
  }
  __device__ void flush() {
    if (n <= 256) return;
    unsigned long long base = 0;
    if ((threadIdx.x & 63) == 0) base = atomicAdd(cursor, (unsigned long long)n);
    write(__shfl(base, 0, 64));
  }
  // The rest of the four waves, by the whole workgroup: one atomic (one of each wave took as long as half
  // the read of the row).
  __device__ void finish(unsigned* counts, unsigned long long* base) {
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) counts[wave] = n;
    __syncthreads();
    const unsigned all = counts[0] + counts[1] + counts[2] + counts[3];
    if (threadIdx.x == 0) *base = all ? atomicAdd(cursor, (unsigned long long)all) : 0ull;
    __syncthreads();
    unsigned long long b = *base;
    for (int w = 0; w < wave; w++) b += counts[w];
    write(b);
  }
};

__device__ inline bool topk_in_row(int64_t i, int64_t count) { return (uint64_t)i < (uint64_t)count; }
// Four entries per lane and turn, of one 16-byte load past the caches, four turns' loads at a time:
// four(their values, the index of the first, whether the whole workgroup's lie in the row; those that do not are zeros, with
// indices that are no entry's).  The turns begin at multiples of 128 bytes wherever the row does, so that no two loads share a
// line (such a line is fetched twice).  10 rows of 12,382,014 entries (every second begins between two pieces of 16 bytes), the
// collection: 4-byte loads 116 to 122 us, now 111; the call at 43 rows of 2,097,023: 168 -> 158.
template <class Four>
__device__ inline void topk_sweep(const float* __restrict__ xr, int64_t count, Four four) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const int64_t step = (int64_t)gridDim.x * 4096;
  const int t = threadIdx.x, before = (int)((uintptr_t)xr >> 2) & 31;
  for (int64_t base = (int64_t)blockIdx.x * 4096 - before; base < count; base += step) {
    if (base >= 0 && base + 4096 <= count) {
      f4 q[4];
#pragma unroll
      for (int u = 0; u < 4; u++)
        q[u] = __builtin_nontemporal_load(reinterpret_cast<const f4*>(xr + (base + 1024 * u + 4 * t)));
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float v[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
        four(v, base + 1024 * u + 4 * t, true);
      }
      continue;
    }
#pragma unroll 1
    for (int64_t b = base; b < base + 4096 && b < count; b += 1024) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int64_t i = b + 4 * t + e;
        v[e] = topk_in_row(i, count) ? xr[i] : 0.0f;
      }
      four(v, b + 4 * t, false);
    }
  }
}

// Fast path: entries whose decided bits are >= the picked prefix (the k-th entry's bin and all
// bins above it) go to the candidate list; the slots past them are padded with the smallest pair.
__global__ void __launch_bounds__(256)
    k_topk_take_bins(const float* __restrict__ x, int64_t count, TopkState* __restrict__ st,
                     uint64_t* __restrict__ cand, int64_t kp, int64_t k) {
  __shared__ uint64_t buf[4][512];
  __shared__ unsigned counts[4];
  __shared__ unsigned long long list_base;
  const int row = blockIdx.y;
  const uint32_t prefix = st[row].prefix, mask = st[row].mask;
  const int64_t n_cand = k - st[row].need + st[row].in_bin;
  uint64_t* out = cand + (int64_t)row * kp;
  topk_finds f{buf[threadIdx.x >> 6], 0u, out, kp, reinterpret_cast<unsigned long long*>(&st[row].cursor), nullptr, nullptr, 0u, 0u, 0, 0};
  topk_sweep(x + (int64_t)row * count, count, [&](const float* v, int64_t first, bool) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const uint32_t key = sort_key(v[e]);
      const int64_t i = first + e;
      f.put(topk_in_row(i, count) && (key & mask) >= prefix, key, i);
    }
    f.flush();
  });
  f.finish(counts, &list_base);
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = n_cand + (int64_t)blockIdx.x * 256 + threadIdx.x; i < kp; i += stride) out[i] = 0;
}

// Entries above T go to the candidate list in any order (the sort fixes it).
__global__ void __launch_bounds__(256)
    k_topk_take_above(const float* __restrict__ x, int64_t count, TopkState* __restrict__ st,
                      uint64_t* __restrict__ cand, int64_t kp) {
  const int row = blockIdx.y;
  const uint32_t T = st[row].prefix;
  const float* xr = x + (int64_t)row * count;
  unsigned long long* cursor = reinterpret_cast<unsigned long long*>(&st[row].cursor);
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += stride) {
    const uint32_t key = sort_key(xr[i]);
    if (key > T) {
      const unsigned long long slot = atomicAdd(cursor, 1ull);
      cand[(int64_t)row * kp + slot] = ((uint64_t)key << 32) | (uint32_t)(0xffffffffu - (uint32_t)i);
    }
  }
}

// Entries equal to T, numbered in index order by `rank` (an exclusive scan of the predicate):
// the first `need` of them complete the list; the slots past k are padded with the smallest pair.
__global__ void __launch_bounds__(256)
    k_topk_take_ties(const float* __restrict__ xr, int64_t count, const TopkState* __restrict__ st_row,
                     const int64_t* __restrict__ rank, uint64_t* __restrict__ cand_row, int64_t k,
                     int64_t kp) {
  const uint32_t T = st_row->prefix;
  const int64_t need = st_row->need, base = k - need;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += stride) {
    if (sort_key(xr[i]) == T && rank[i] < need)
      cand_row[base + rank[i]] = ((uint64_t)T << 32) | (uint32_t)(0xffffffffu - (uint32_t)i);
  }
  for (int64_t i = k + (int64_t)blockIdx.x * 256 + threadIdx.x; i < kp; i += stride) cand_row[i] = 0;
}

struct TieF {
  const float* x;
  const TopkState* st;
  __device__ int64_t operator()(int64_t i) const { return sort_key(x[i]) == st->prefix ? 1 : 0; }
};

// ---- bitonic sort, descending, of kp (a power of two) pairs per row ----
constexpr int BITONIC_CHUNK = 4096;

__device__ inline void cmp_swap_desc(uint64_t& a, uint64_t& b, bool descending) {
  if ((a < b) == descending) {
    const uint64_t t = a;
    a = b;
    b = t;
  }
}

// All merge steps with stride < BITONIC_CHUNK of the stages size_lo .. size_hi, inside LDS.
__global__ void __launch_bounds__(256)
    k_bitonic_local(uint64_t* __restrict__ data, int64_t kp, int64_t size_lo, int64_t size_hi) {
  __shared__ uint64_t s[BITONIC_CHUNK];
  uint64_t* d = data + (int64_t)blockIdx.y * kp + (int64_t)blockIdx.x * BITONIC_CHUNK;
  const int64_t g0 = (int64_t)blockIdx.x * BITONIC_CHUNK;
  const int n = kp < BITONIC_CHUNK ? (int)kp : BITONIC_CHUNK;
  for (int i = threadIdx.x; i < n; i += 256) s[i] = d[i];
  __syncthreads();
  for (int64_t size = size_lo; size <= size_hi; size <<= 1) {
    int64_t j = size >> 1;
    if (j >= BITONIC_CHUNK) j = BITONIC_CHUNK >> 1;
    for (; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < n / 2; t += 256) {
        const int lo = (int)(((int64_t)t / j) * 2 * j + t % j), hi = lo + (int)j;
        const bool desc = ((g0 + lo) & size) == 0;
        cmp_swap_desc(s[lo], s[hi], desc);
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < n; i += 256) d[i] = s[i];
}

// One merge step with stride j >= BITONIC_CHUNK of stage `size`.
__global__ void __launch_bounds__(256)
    k_bitonic_global(uint64_t* __restrict__ data, int64_t kp, int64_t size, int64_t j) {
  uint64_t* d = data + (int64_t)blockIdx.y * kp;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < kp / 2; t += stride) {
    const int64_t lo = (t / j) * 2 * j + t % j, hi = lo + j;
    uint64_t a = d[lo], b = d[hi];
    cmp_swap_desc(a, b, (lo & size) == 0);
    d[lo] = a;
    d[hi] = b;
  }
}

__global__ void __launch_bounds__(256)
    k_topk_emit(const uint64_t* __restrict__ cand, int64_t k, int64_t kp, float* __restrict__ vals,
                int32_t* __restrict__ idx) {
  const int row = blockIdx.y;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < k; i += stride) {
    const uint64_t c = cand[(int64_t)row * kp + i];
    vals[(int64_t)row * k + i] = key_to_float((uint32_t)(c >> 32));
    idx[(int64_t)row * k + i] = (int32_t)(0xffffffffu - (uint32_t)c);
  }
}

// ---------------------------------------------------------------------------
// The usual case
// ---------------------------------------------------------------------------
struct TopkRow {
  uint32_t bin, thr, top;      // top: the largest key of the sample
  unsigned need;               // of the sample, still to find
  unsigned long long cursor;   // candidates
};

__global__ void __launch_bounds__(1024)
    k_topk_row_init(TopkRow* rows, unsigned target, unsigned* __restrict__ hist, int nb, int* __restrict__ buckets) {
  if (threadIdx.x == 0) rows[blockIdx.x] = TopkRow{0u, 0u, 0u, target, 0ull};
  for (int i = threadIdx.x; i < TOPK_BINS; i += 1024) hist[(int64_t)blockIdx.x * TOPK_BINS + i] = 0;
  for (int i = threadIdx.x; i < nb; i += 1024) buckets[(int64_t)blockIdx.x * nb + i] = 0;
}

// A workgroup of 16 waves and two rounds of loads per wave (128 chunks): every workgroup adds its histogram to the row's few
// busy lines, and it is those additions that wait for each other.  2 rows of 110 M, LEVEL 0: 8.7 us; 16.3 with workgroups
// of four waves and 64 chunks, 10.9 with 512 chunks for 16 waves.
constexpr int TOPK_SAMPLE_WAVES = 16;
constexpr int TOPK_SAMPLE_EACH = 128;
// LEVEL 0: top 11 bits of the key, and the largest key; 1: the next 11 of the entries in the bin that level 0 found.
template <int LEVEL>
__global__ void __launch_bounds__(TOPK_SAMPLE_WAVES * 64)
    k_topk_sample(const float* __restrict__ x, int64_t count, int64_t stride, int64_t chunks,
                  TopkRow* __restrict__ rows, unsigned* __restrict__ hist) {
  __shared__ unsigned h[TOPK_BINS];
  __shared__ uint32_t most[TOPK_SAMPLE_WAVES];
  const int row = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int i = threadIdx.x; i < TOPK_BINS; i += TOPK_SAMPLE_WAVES * 64) h[i] = 0;
  const uint32_t bin = LEVEL ? rows[row].bin : 0u;
  uint32_t top = 0;
  __syncthreads();
  const float* xr = x + (int64_t)row * count;
  const int64_t step = (int64_t)gridDim.x * TOPK_SAMPLE_WAVES;
  for (int64_t c = (int64_t)blockIdx.x * TOPK_SAMPLE_WAVES + wave; c < chunks; c += 4 * step) {
    float v[4];
    bool ok[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int64_t i = (c + u * step) * stride + lane;
      ok[u] = c + u * step < chunks && i < count;
      v[u] = xr[ok[u] ? i : 0];
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const uint32_t key = sort_key(v[u]);
      if (LEVEL) ok[u] = ok[u] && (key >> 21) == bin;
      else top = ok[u] ? max(top, key) : top;
      if (ok[u]) atomicAdd(&h[LEVEL ? (key >> 10) & (TOPK_BINS - 1) : key >> 21], 1u);
    }
  }
  if (!LEVEL) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, off));
    if (lane == 0) most[wave] = top;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < TOPK_BINS; i += TOPK_SAMPLE_WAVES * 64)
    if (h[i]) atomicAdd(&hist[(int64_t)row * TOPK_BINS + i], h[i]);
  if (!LEVEL && threadIdx.x == 0) {
    for (int w = 1; w < TOPK_SAMPLE_WAVES; w++) top = max(top, most[w]);
    atomicMax(&rows[row].top, top);
  }
}

// The bin from the top where the sample's entries reach the target.
template <int LEVEL>
__global__ void __launch_bounds__(256) k_topk_threshold(unsigned* __restrict__ hist, TopkRow* __restrict__ rows) {
  __shared__ unsigned part[256];
  unsigned* h = hist + (int64_t)blockIdx.x * TOPK_BINS;
  const int t = threadIdx.x, top = TOPK_BINS - 1 - 8 * t;  // thread t: eight bins from `top` down
  unsigned c[8], sum = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) sum += c[i] = h[top - i];
  part[t] = sum;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const unsigned add = t >= off ? part[t - off] : 0;
    __syncthreads();
    part[t] += add;
    __syncthreads();
  }
  const unsigned need = rows[blockIdx.x].need, total = part[255];
  unsigned above = part[t] - sum;
  __syncthreads();
  if (above < need && above + sum >= need) {
    int b = 0;
    while (above + c[b] < need) above += c[b++];
    TopkRow& r = rows[blockIdx.x];
    if (LEVEL == 0) {
      r.bin = (uint32_t)(top - b);
      r.need = need - above;
    } else {
      r.thr = (r.bin << 21) | ((uint32_t)(top - b) << 10);
    }
  }
  if (t == 0 && total < need) {  // (fewer entries than the target: everything is a candidate)
    rows[blockIdx.x].bin = 0;
    rows[blockIdx.x].thr = 0;
  }
  __syncthreads();
  if (LEVEL == 0)
    for (int i = t; i < TOPK_BINS; i += 256) h[i] = 0;
}

// Both levels of a row of few chunks by one workgroup: what five launches (the start, two histograms and their bins) else take.
// 64 rows of 20,000: 72 -> 48 us a call, 1 of 16,000 71 -> 42, 3 of 1,000,000 (489 chunks) 73 -> 55, 40 of 700,000 86 -> 74. Past
// 512 chunks it falls behind: 20 of 60,000 (938) 66 us against 54, 5 of 4,000,000 (1954) 174 against 147.
constexpr int TOPK_SHORT = 512;
__global__ void __launch_bounds__(1024)
    k_topk_short(const float* __restrict__ x, int64_t count, int64_t stride, int64_t chunks, unsigned target,
                 TopkRow* __restrict__ rows, int* __restrict__ buckets, int nb) {
  static_assert(TOPK_BINS == 2 * 1024, "a thread has two bins");
  __shared__ unsigned h[TOPK_BINS];
  __shared__ unsigned part[16];
  __shared__ uint32_t most[16], found_bin, found_need;
  const int row = blockIdx.x, t = threadIdx.x, wave = t >> 6, lane = t & 63;
  for (int i = t; i < nb; i += 1024) buckets[(int64_t)row * nb + i] = 0;
  const float* xr = x + (int64_t)row * count;
  uint32_t bin = 0, thr = 0, top = 0;
  unsigned need = target;
  for (int level = 0; level < 2; level++) {
    h[t] = h[t + 1024] = 0;
    __syncthreads();
    constexpr int U = 8;
    for (int64_t c = wave; c < chunks; c += 16 * U) {
      float v[U];
      bool ok[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int64_t i = (c + 16 * u) * stride + lane;
        ok[u] = c + 16 * u < chunks && i < count;
        v[u] = xr[ok[u] ? i : 0];
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint32_t key = sort_key(v[u]);
        if (level) ok[u] = ok[u] && (key >> 21) == bin;
        else top = ok[u] ? max(top, key) : top;
        if (ok[u]) atomicAdd(&h[level ? (key >> 10) & (TOPK_BINS - 1) : key >> 21], 1u);
      }
    }
    if (level == 0) {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, off));
      if (lane == 0) most[wave] = top;
    }
    __syncthreads();
    // the bin from the top where the entries reach the target: thread t has bins 2047 - 2 t and the one below
    const int first = TOPK_BINS - 1 - 2 * t;
    const unsigned c0 = h[first], c1 = h[first - 1];
    unsigned incl = c0 + c1;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned up = __shfl_up(incl, off);
      if (lane >= off) incl += up;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    unsigned total = 0, above = incl - (c0 + c1);
    for (int w = 0; w < 16; w++) {
      if (w < wave) above += part[w];
      total += part[w];
    }
    if (above < need && above + c0 + c1 >= need) {
      const int b = above + c0 < need;
      found_bin = (uint32_t)(first - b);
      found_need = need - above - (b ? c0 : 0u);
    }
    __syncthreads();
    const bool all = total < need;  // (fewer entries than the target: everything is a candidate)
    if (level == 0) {
      bin = all ? 0u : found_bin;
      need = all ? need : found_need;
    } else {
      thr = all ? 0u : (bin << 21) | (found_bin << 10);
    }
    __syncthreads();
  }
  if (t == 0) {
    for (int w = 0; w < 16; w++) top = max(top, most[w]);
    rows[row] = TopkRow{bin, thr, top, need, 0ull};
  }
}

// Entries from the threshold up and the sum of squares.  Bound by the read of the row (2 rows of
// 110 M: 145 to 154 us, 5.7 to 6.1 TB/s; a barrier and a shared buffer per 1024 entries: 200 us).
__global__ void __launch_bounds__(256)
    k_topk_collect(const float* __restrict__ x, int64_t count, TopkRow* __restrict__ rows, uint64_t* __restrict__ cand,
                   int64_t cap, int log_nb, int above, int* __restrict__ buckets, unsigned* __restrict__ place,
                   double* __restrict__ sq_partials) {
  __shared__ uint64_t buf[4][512];
  __shared__ unsigned counts[4];
  __shared__ unsigned long long list_base;
  __shared__ double red[256];
  const int row = blockIdx.y;
  const uint32_t thr = rows[row].thr, top = rows[row].top;
  topk_finds f{buf[threadIdx.x >> 6], 0u, cand + (int64_t)row * cap, cap, &rows[row].cursor,
               buckets + (int64_t)row * ((1 << log_nb) + above), place + (int64_t)row * cap, thr, top, topk_shift(thr, top, log_nb), above};
  double sq = 0.0;
  // (from the key of +0 up, keys are in the order of the bits as signed integers)
  const bool plain = thr >= 0x80000000u;
  const int thr_bits = (int)(thr & 0x7fffffffu);
  topk_sweep(x + (int64_t)row * count, count, [&](const float* v, int64_t first, bool whole) {
    bool any = true;
    if (whole) {
#pragma unroll
      for (int e = 0; e < 4; e++) sq += (double)v[e] * (double)v[e];
      if (plain)
        any = max(max(__float_as_int(v[0]), __float_as_int(v[1])), max(__float_as_int(v[2]), __float_as_int(v[3]))) >=
              thr_bits;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (topk_in_row(first + e, count)) sq += (double)v[e] * (double)v[e];
    }
    if (__any(any)) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t key = sort_key(v[e]);
        const int64_t i = first + e;
        const bool take = topk_in_row(i, count) && key >= thr;
        f.put(take, key, i);
      }
      f.flush();
    }
  });
  f.finish(counts, &list_base);
  red[threadIdx.x] = sq;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) sq_partials[(int64_t)row * gridDim.x + blockIdx.x] = red[0];
}

// Counts to starts (in place), the row's norm, and whether the list serves.
// (A row has one workgroup here, so a thread has at most 20 counts and loads them four at a time, and sums go
// by shuffles: 16,384 counts, 2 rows, 6.3 us; 9.5 with ten barriers, 43 with 64 counts one at a time.)
constexpr int TOPK_SCAN = 1024;
__global__ void __launch_bounds__(TOPK_SCAN)
    k_topk_bucket_scan(const TopkRow* __restrict__ rows, int64_t cap, int64_t k, int nb, int* __restrict__ buckets,
                       const double* __restrict__ sq_partials, int n_sq,
                       float* __restrict__ norms, unsigned long long* __restrict__ failed) {
  __shared__ int part[TOPK_SCAN / 64];
  __shared__ double red[TOPK_SCAN / 64];
  const int row = blockIdx.x, t = threadIdx.x, quads = (nb / 4 + TOPK_SCAN - 1) / TOPK_SCAN;
  int4* b = reinterpret_cast<int4*>(buckets + (int64_t)row * nb);
  constexpr int MOST = TOPK_MAX_BUCKETS / 4 / TOPK_SCAN;
  const int mine = min(quads, max(0, nb / 4 - t * quads));
  int4 v[MOST];
  int sum = 0, most = 0;
#pragma unroll
  for (int i = 0; i < MOST; i++) {
    v[i] = i < mine ? b[t * quads + i] : int4{0, 0, 0, 0};
    sum += v[i].x + v[i].y + v[i].z + v[i].w;
    most = max(max(max(v[i].x, v[i].y), max(v[i].z, v[i].w)), most);
  }
  double s = 0.0;
  for (int i = t; i < n_sq; i += TOPK_SCAN) s += sq_partials[(int64_t)row * n_sq + i];
  const int wave = t >> 6, lane = t & 63;
  int incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int up = __shfl_up(incl, off);
    if (lane >= off) incl += up;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (lane == 63) part[wave] = incl;
  if (lane == 0) red[wave] = s;
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wave; w++) run += part[w];
#pragma unroll
  for (int i = 0; i < MOST; i++) {
    if (i >= mine) break;
    const int4 w{run, run + v[i].x, run + v[i].x + v[i].y, run + v[i].x + v[i].y + v[i].z};
    b[t * quads + i] = w;
    run = w.w + v[i].w;
  }
  if (t == 0) {
    for (int w = 1; w < TOPK_SCAN / 64; w++) s += red[w];
    if (norms) norms[row] = (float)sqrt(s);
    if ((int64_t)rows[row].cursor < k || (int64_t)rows[row].cursor > cap) *failed = 1;
  }
  if (most > TOPK_CROWDED) *failed = 1;
}

__global__ void __launch_bounds__(256)
    k_topk_scatter(const TopkRow* __restrict__ rows, const uint64_t* __restrict__ cand, const unsigned* __restrict__ place,
                   int64_t cap, int log_nb, int above, const int* __restrict__ starts, uint64_t* __restrict__ out) {
  const TopkRow r = rows[blockIdx.y];
  const int64_t n = (int64_t)r.cursor < cap ? (int64_t)r.cursor : cap;
  const int shift = topk_shift(r.thr, r.top, log_nb);
  const int* s = starts + (int64_t)blockIdx.y * ((1 << log_nb) + above);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const uint64_t p = cand[(int64_t)blockIdx.y * cap + i];
    out[(int64_t)blockIdx.y * cap + s[topk_bucket((uint32_t)(p >> 32), r.thr, r.top, shift, above)] + place[(int64_t)blockIdx.y * cap + i]] = p;
  }
}

// The k first places: a pair's is its bucket's start plus the larger pairs of the bucket.
__global__ void __launch_bounds__(256)
    k_topk_rank(const TopkRow* __restrict__ rows, const uint64_t* __restrict__ sorted, int64_t cap, int64_t k, int log_nb,
                int above, const int* __restrict__ starts, float* __restrict__ vals,
                int32_t* __restrict__ idx) {
  const TopkRow r = rows[blockIdx.y];
  const int64_t n = (int64_t)r.cursor < cap ? (int64_t)r.cursor : cap;
  const int shift = topk_shift(r.thr, r.top, log_nb);
  const uint64_t* p = sorted + (int64_t)blockIdx.y * cap;
  const int nb = (1 << log_nb) + above;
  const int* row_starts = starts + (int64_t)blockIdx.y * nb;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const uint64_t own = p[i];
    const int b = topk_bucket((uint32_t)(own >> 32), r.thr, r.top, shift, above);
    const int s = row_starts[b], e = b + 1 < nb ? row_starts[b + 1] : (int)n;
    if (s >= k || e - s > TOPK_CROWDED) continue;
    int rank = s;
    for (int j = s; j < e; j++) rank += p[j] > own;
    if (rank < k) {
      vals[(int64_t)blockIdx.y * k + rank] = key_to_float((uint32_t)(own >> 32));
      idx[(int64_t)blockIdx.y * k + rank] = (int32_t)(0xffffffffu - (uint32_t)own);
    }
  }
}

}  // namespace dn

using namespace dn;

// Candidate lists longer than this (k plus the k-th entry's bin) take the exact-threshold path.
constexpr int64_t TOPK_FAST_CAP = (int64_t)1 << 21;

static int bitonic_sort_rows(uint64_t* cand, int64_t kp, int64_t n_rows) {
  hipStream_t st = stream();
  const dim3 block(256);
  const unsigned chunks = (unsigned)ceil_div(kp, BITONIC_CHUNK);
  const int64_t local_hi = kp < BITONIC_CHUNK ? kp : BITONIC_CHUNK;
  hipLaunchKernelGGL(k_bitonic_local, dim3(chunks, (unsigned)n_rows), block, 0, st, cand, kp, (int64_t)2,
                     local_hi);
  unsigned gg = (unsigned)ceil_div(kp / 2, 256);
  if (gg > 4096) gg = 4096;
  if (gg < 1) gg = 1;
  for (int64_t size = 2 * (int64_t)BITONIC_CHUNK; size <= kp; size <<= 1) {
    for (int64_t j = size >> 1; j >= BITONIC_CHUNK; j >>= 1)
      hipLaunchKernelGGL(k_bitonic_global, dim3(gg, (unsigned)n_rows), block, 0, st, cand, kp, size, j);
    hipLaunchKernelGGL(k_bitonic_local, dim3(chunks, (unsigned)n_rows), block, 0, st, cand, kp, size, size);
  }
  DN_LAUNCH_CHECK();
  return 0;
}

// Results on their way to the host (dnpeff_topk_rows_host).
struct topk_down {
  static constexpr int BUFS = 2;
  copy_part parts[3];
  int n_parts;
  pinned_buf pinned[BUFS];
  copy_part of[BUFS][3];  // what goes through which: of each array one piece at most
  int n_of[BUFS] = {};
  bool queued = false;

  // Where two pinned buffers hold them, they go there behind the last kernel, before it is known whether that served;
  // and the pages of the host's arrays, which a first write would have to fetch between the results and the
  // return, are fetched while the device works.
  int queue() {
    int b = 0;
    size_t used = 0;
    for (int q = 0; q < n_parts; q++)
      for (size_t off = 0; off < parts[q].bytes;) {
        if (used + 16 > pinned_buf::BYTES) {
          if (++b == BUFS) return 0;
          used = 0;
        }
        const size_t left = parts[q].bytes - off, room = (pinned_buf::BYTES - used) / 16 * 16, n = left < room ? left : room;
        of[b][n_of[b]++] = {(char*)parts[q].dst + off, (const char*)parts[q].src + off, n};
        used += gather_room(n);
        off += n;
      }
    for (int i = 0; i <= b; i++) {
      pinned[i].take();
      if (!pinned[i].p()) return 0;
    }
    for (int i = 0; i <= b; i++) DN_HIP(gather_queue(of[i], n_of[i], pinned[i].p()));
    queued = true;
    for (int q = 0; q < n_parts; q++) fetch_pages(parts[q].dst, parts[q].bytes);
    return 0;
  }
  void take() {
    for (int i = 0; i < BUFS; i++) gather_take(of[i], n_of[i], pinned[i].p());
  }
};

// The usual case; *done = false: a row needs the histograms of all entries.
static int topk_by_sample(int64_t n_rows, int64_t count, int64_t k, const float* x, float* vals, int32_t* idx,
                          float* norms, topk_down* down, bool* done) {
  *done = false;
  const topk_plan plan = topk_plan_of(count, k);
  const int64_t stride = plan.stride, chunks = ceil_div(count, stride), cap = plan.cap;
  const int log_nb = plan.log_nb, above = plan.above;
  if ((double)n_rows * (double)cap * 16.0 > 4.0e9) return 0;
  hipStream_t st = stream();
  const dim3 block(256);
  // (one launch fills the chip several times over, however many rows there are)
  const int64_t most = std::max<int64_t>(8, 2048 / n_rows);
  auto blocks = [&](int64_t items, int64_t each) {
    const int64_t g = ceil_div(items, each);
    return dim3((unsigned)std::max<int64_t>(1, std::min(g, most)), (unsigned)n_rows);
  };
  dbuf<TopkRow> rows;
  dbuf<unsigned> hist;
  dbuf<uint64_t> cand, sorted;
  dbuf<int> starts;
  dbuf<unsigned> place;
  dbuf<double> sq;
  const dim3 gc = blocks(count, 4096);
  DN_TRY(rows.alloc(n_rows));
  DN_TRY(cand.alloc(n_rows * cap));
  DN_TRY(sorted.alloc(n_rows * cap));
  DN_TRY(starts.alloc(n_rows * plan.buckets()));
  DN_TRY(place.alloc(n_rows * cap));
  DN_TRY(sq.alloc(n_rows * gc.x));
  unsigned long long* failed = nullptr;
  DN_TRY(host_words(&failed));
  *failed = 0;
  const dim3 gs = blocks(chunks, TOPK_SAMPLE_EACH), gr((unsigned)n_rows), gp = blocks(cap, 256);
  if (chunks <= TOPK_SHORT) {
    hipLaunchKernelGGL(k_topk_short, gr, dim3(1024), 0, st, x, count, stride, chunks, plan.target, rows.p, starts.p, plan.buckets());
  } else {
    DN_TRY(hist.alloc(n_rows * TOPK_BINS));
    hipLaunchKernelGGL(k_topk_row_init, gr, dim3(1024), 0, st, rows.p, plan.target, hist.p, plan.buckets(), starts.p);
    hipLaunchKernelGGL(k_topk_sample<0>, gs, dim3(TOPK_SAMPLE_WAVES * 64), 0, st, x, count, stride, chunks, rows.p, hist.p);
    hipLaunchKernelGGL(k_topk_threshold<0>, gr, block, 0, st, hist.p, rows.p);
    hipLaunchKernelGGL(k_topk_sample<1>, gs, dim3(TOPK_SAMPLE_WAVES * 64), 0, st, x, count, stride, chunks, rows.p, hist.p);
    hipLaunchKernelGGL(k_topk_threshold<1>, gr, block, 0, st, hist.p, rows.p);
  }
  hipLaunchKernelGGL(k_topk_collect, gc, block, 0, st, x, count, rows.p, cand.p, cap, log_nb, above, starts.p, place.p, sq.p);
  hipLaunchKernelGGL(k_topk_bucket_scan, gr, dim3(TOPK_SCAN), 0, st, rows.p, cap, k, plan.buckets(), starts.p, sq.p, (int)gc.x,
                     norms, failed);
  hipLaunchKernelGGL(k_topk_scatter, gp, block, 0, st, rows.p, cand.p, place.p, cap, log_nb, above, starts.p, sorted.p);
  hipLaunchKernelGGL(k_topk_rank, gp, block, 0, st, rows.p, sorted.p, cap, k, log_nb, above, starts.p, vals, idx);
  DN_LAUNCH_CHECK();
  const int q = down ? down->queue() : 0;
  DN_HIP(hipStreamSynchronize(st));
  DN_TRY(q);
  *done = *failed == 0;
  return 0;
}

static int topk_check(int64_t n_rows, int64_t count, int64_t k, const float* x, const float* vals_out,
                      const int32_t* idx_out) {
  DN_CHECK(n_rows >= 0 && n_rows <= 65535, "n_rows %lld outside [0, 65535]", (long long)n_rows);
  DN_CHECK(count >= 1 && count <= (int64_t)INT32_MAX, "count %lld outside [1, 2^31)", (long long)count);
  DN_CHECK(k >= 1 && k <= count && k <= ((int64_t)1 << 24), "k %lld outside [1, min(count, 2^24)]",
           (long long)k);
  DN_CHECK(x && vals_out && idx_out, "NULL argument");
  return 0;
}

static int topk_of_rows(int64_t n_rows, int64_t count, int64_t k, const float* x, float* vals_out, int32_t* idx_out,
                        float* norms_out, topk_down* down) {
  if (n_rows == 0) return 0;
  if (tuning().topk_fast_cap < 0.0) {  // (tests force the deeper paths)
    bool done = false;
    DN_TRY(topk_by_sample(n_rows, count, k, x, vals_out, idx_out, norms_out, down, &done));
    if (done) return 0;
    if (down) down->queued = false;
  }
  hipStream_t st = stream();
  unsigned gx = (unsigned)ceil_div(count, 256 * 16);
  if (gx > 2048) gx = 2048;
  if (gx < 1) gx = 1;
  const dim3 grid(gx, (unsigned)n_rows), block(256);
  TopkState* state = nullptr;
  unsigned* hist = nullptr;
  uint64_t* cand = nullptr;
  int64_t* rank = nullptr;
  double* sq = nullptr;
  auto cleanup = [&]() {
    (void)hipStreamSynchronize(st);
    dfree(state); dfree(hist); dfree(cand); dfree(rank); dfree(sq);
  };
  int s = dmalloc(&state, n_rows) || dmalloc(&hist, n_rows * TOPK_BINS) || dmalloc(&sq, n_rows * gx);
  if (!s && hipMemsetAsync(hist, 0, sizeof(unsigned) * n_rows * TOPK_BINS, st) != hipSuccess) {
    set_error("top-k: clearing the histograms failed");
    s = 1;
  }
  if (s) { cleanup(); return s; }
  hipLaunchKernelGGL(k_topk_init, dim3((unsigned)n_rows), dim3(1), 0, st, state, k);
  const bool vec4 = count % 4 == 0 && ((uintptr_t)x % 16) == 0;
  auto launch_hist = [&](int shift, int nbits, double* sq_out) {
    if (vec4)
      hipLaunchKernelGGL(k_topk_hist<true>, grid, block, 0, st, x, count, shift, nbits, state, hist, sq_out);
    else
      hipLaunchKernelGGL(k_topk_hist<false>, grid, block, 0, st, x, count, shift, nbits, state, hist, sq_out);
  };
  launch_hist(21, 11, sq);
  hipLaunchKernelGGL(k_topk_pick, dim3((unsigned)n_rows), dim3(64), 0, st, hist, 21, 11, state);
  if (norms_out)
    hipLaunchKernelGGL(k_topk_norm, dim3((unsigned)n_rows), dim3(64), 0, st, sq, (int)gx, norms_out);
  std::vector<TopkState> host_state((size_t)n_rows);
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess ||
      copy_down(host_state.data(), state, sizeof(TopkState) * n_rows) != hipSuccess) {
    set_error("top-k: the first pass failed");
    cleanup();
    return 1;
  }
  auto longest_list = [&]() {
    int64_t most = 0;
    for (const TopkState& h : host_state) {
      const int64_t n_cand = k - h.need + h.in_bin;
      if (n_cand > most) most = n_cand;
    }
    return most;
  };
  int64_t kp = 1, cap = TOPK_FAST_CAP;
  if (tuning().topk_fast_cap >= 0.0) cap = (int64_t)tuning().topk_fast_cap;  // tests: force the deeper paths
  // while the k-th entry's bin is crowded, decide the next bits of the key (one more read each)
  const int shifts[2] = {10, 0}, bits[2] = {11, 10};
  int64_t most = longest_list();
  for (int p = 0; p < 2 && most > cap; p++) {
    launch_hist(shifts[p], bits[p], nullptr);
    hipLaunchKernelGGL(k_topk_pick, dim3((unsigned)n_rows), dim3(64), 0, st, hist, shifts[p], bits[p], state);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess ||
        copy_down(host_state.data(), state, sizeof(TopkState) * n_rows) != hipSuccess) {
      set_error("top-k: a histogram pass failed");
      cleanup();
      return 1;
    }
    most = longest_list();
  }
  if (most <= cap) {
    while (kp < most) kp <<= 1;
    s = dmalloc(&cand, n_rows * kp);
    if (!s) {
      hipLaunchKernelGGL(k_topk_take_bins, grid, block, 0, st, x, count, state, cand, kp, k);
      s = bitonic_sort_rows(cand, kp, n_rows);
    }
  } else {
    // the whole key is decided and the entries equal to it alone are too many to sort: take
    // the first `need` of them in index order
    while (kp < k) kp <<= 1;
    s = dmalloc(&cand, n_rows * kp) || dmalloc(&rank, count + 1);
    if (!s) {
      hipLaunchKernelGGL(k_topk_take_above, grid, block, 0, st, x, count, state, cand, kp);
      if (hipGetLastError() != hipSuccess) { set_error("top-k: launch failed"); s = 1; }
    }
    for (int64_t row = 0; row < n_rows && !s; row++) {
      const float* xr = x + row * count;
      s = exclusive_scan(TieF{xr, state + row}, count, rank);
      if (!s)
        hipLaunchKernelGGL(k_topk_take_ties, dim3(gx), block, 0, st, xr, count, state + row, rank,
                           cand + row * kp, k, kp);
    }
    if (!s) s = bitonic_sort_rows(cand, kp, n_rows);
  }
  if (!s) {
    unsigned ge = (unsigned)ceil_div(k, 256);
    if (ge > 4096) ge = 4096;
    hipLaunchKernelGGL(k_topk_emit, dim3(ge, (unsigned)n_rows), block, 0, st, cand, k, kp, vals_out, idx_out);
    if (hipGetLastError() != hipSuccess) { set_error("top-k: launch failed"); s = 1; }
  }
  cleanup();
  return s;
}

DN_API int dnpeff_topk_rows(int64_t n_rows, int64_t count, int64_t k, const float* x, float* vals_out,
                            int32_t* idx_out, float* norms_out) {
  clear_error();
  DN_TRY(topk_check(n_rows, count, k, x, vals_out, idx_out));
  return topk_of_rows(n_rows, count, k, x, vals_out, idx_out, norms_out, nullptr);
}

// 2 rows of 110 M, k = 65,536: 291 us with dnpeff_topk_rows, its wait and a download behind it, 277 this way.  10 rows of 12.4 M, k =
// 38,482 (3 MB), into arrays that are new: 850 us, now 560.
DN_API int dnpeff_topk_rows_host(int64_t n_rows, int64_t count, int64_t k, const float* x, float* vals_host,
                                 int32_t* idx_host, float* norms_host) {
  clear_error();
  DN_TRY(topk_check(n_rows, count, k, x, vals_host, idx_host));
  dbuf<float> vals, norms;
  dbuf<int32_t> idx;
  const size_t n = (size_t)(n_rows * k);
  DN_TRY(vals.alloc((int64_t)n));
  DN_TRY(idx.alloc((int64_t)n));
  if (norms_host) DN_TRY(norms.alloc(n_rows));
  topk_down down{{{vals_host, vals.p, 4 * n}, {idx_host, idx.p, 4 * n}, {norms_host, norms.p, 4 * (size_t)n_rows}},
                 norms_host ? 3 : 2};
  DN_TRY(topk_of_rows(n_rows, count, k, x, vals.p, idx.p, norms.p, &down));
  if (n_rows == 0) return 0;
  if (down.queued) down.take();
  else DN_HIP(copy_down_parts(down.parts, down.n_parts));
  return 0;
}
