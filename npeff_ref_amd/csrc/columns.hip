// Dropping columns: which are kept is one bit each, the new number of a column is a rank.
//
// A column's bit and the ranks of the bits' words together take a sixteenth of what a table of column
// numbers takes (11 M columns: 2.8 MB instead of 44), so the two random lookups per entry stay in an
// XCD's L2, and the scans over the columns shrink by the same factor.
#include "dnpeff_internal.hpp"
#include "scan.hpp"

#include <algorithm>

namespace dn {

constexpr int MARK_THREADS = 1024;
constexpr int MARK_LDS_WORDS = 32768;  // 128 KB of marks per workgroup
constexpr int KEPT_TILE = 4096;        // entries per workgroup of the passes over the entries

// Marks of the columns of one range (blockIdx.x) from one part of the entries (blockIdx.y): a bit that is
// set by the first entry of a column, for TWO another that the second sets.  out[range][part][plane][word].
// Sixteen million counter updates in memory run at 20 G/s whatever the columns are (760 us); in LDS they
// cost little, and the column numbers, read once for every half a million columns (22 times), come out of
// the memory-side cache: 16.4 M entries, 11 M columns: 175 us.
template <bool TWO>
__global__ void __launch_bounds__(MARK_THREADS)
    k_mark_columns(const int32_t* __restrict__ colind, int64_t nnz, int64_t per_part, int words,
                   uint32_t* __restrict__ out) {
  extern __shared__ uint32_t marks[];
  uint32_t* one = marks;
  uint32_t* two = marks + words;
  const int n = TWO ? 2 * words : words;
  for (int i = threadIdx.x; i < n; i += MARK_THREADS) marks[i] = 0;
  __syncthreads();
  const unsigned lo = (unsigned)blockIdx.x * 32u * (unsigned)words, span = 32u * (unsigned)words;
  auto mark = [&](int32_t col) {
    const unsigned c = (unsigned)col - lo;
    if (c >= span) return;
    const uint32_t bit = 1u << (c & 31);
    if (TWO) {
      if (atomicOr(&one[c >> 5], bit) & bit) atomicOr(&two[c >> 5], bit);
    } else {
      atomicOr(&one[c >> 5], bit);
    }
  };
  const int64_t e0 = (int64_t)blockIdx.y * per_part, e1 = e0 + per_part < nnz ? e0 + per_part : nnz;
  constexpr int STEP = 4 * MARK_THREADS;
  int64_t e = e0 + 4 * threadIdx.x;
  for (; e + STEP + 3 < e1; e += 2 * STEP) {  // (per_part is a multiple of 4)
    const int4 a = *reinterpret_cast<const int4*>(colind + e), b = *reinterpret_cast<const int4*>(colind + e + STEP);
    mark(a.x); mark(a.y); mark(a.z); mark(a.w);
    mark(b.x); mark(b.y); mark(b.z); mark(b.w);
  }
  for (; e < e1; e += STEP)
    for (int u = 0; u < 4; u++)
      if (e + u < e1) mark(colind[e + u]);
  __syncthreads();
  uint32_t* dst = out + ((int64_t)blockIdx.x * gridDim.y + blockIdx.y) * n;
  for (int i = threadIdx.x; i < n; i += MARK_THREADS) dst[i] = marks[i];
}

// The parts' marks together: columns with an entry, for TWO with two.
template <bool TWO>
__global__ void __launch_bounds__(256)
    k_merge_marks(const uint32_t* __restrict__ marks, int parts, int words, int64_t n_words, uint32_t* __restrict__ mask) {
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= n_words) return;
  const int64_t range = w / words;
  const int n = TWO ? 2 * words : words;
  const uint32_t* m = marks + range * parts * n + w % words;
  uint32_t one = 0, two = 0;
  for (int p = 0; p < parts; p++) {
    const uint32_t a = m[(int64_t)p * n];
    if (TWO) two |= m[(int64_t)p * n + words] | (one & a);
    one |= a;
  }
  mask[w] = TWO ? two : one;
}

// Columns with min_count entries or more.
__global__ void __launch_bounds__(256)
    k_mask_of_counts(const int* __restrict__ count, int min_count, int64_t n_cols, int64_t n_words,
                     uint32_t* __restrict__ mask) {
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= n_words) return;
  uint32_t bits = 0;
  for (int b = 0; b < 32; b++)
    if (32 * w + b < n_cols && count[32 * w + b] >= min_count) bits |= 1u << b;
  mask[w] = bits;
}

// The columns of an ascending list.
__global__ void __launch_bounds__(256)
    k_mask_of_list(const int32_t* __restrict__ kept, int64_t n_kept, int64_t n_words, uint32_t* __restrict__ mask) {
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= n_words) return;
  int64_t a = 0, b = n_kept;
  while (a < b) {
    const int64_t mid = (a + b) >> 1;
    if (kept[mid] < 32 * w) a = mid + 1;
    else b = mid;
  }
  uint32_t bits = 0;
  for (; a < n_kept && kept[a] < 32 * w + 32; a++) bits |= 1u << (kept[a] & 31);
  mask[w] = bits;
}

// new_to_og[rank of i] = i
__global__ void __launch_bounds__(256)
    k_list_of_mask(const uint32_t* __restrict__ mask, const int32_t* __restrict__ rank, int64_t n_words,
                   int32_t* __restrict__ new_to_og) {
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= n_words) return;
  int32_t at = rank[w];
  for (uint32_t bits = mask[w]; bits; bits &= bits - 1) new_to_og[at++] = (int32_t)(32 * w) + __ffs((int)bits) - 1;
}

struct MaskBitsF {
  const uint32_t* mask;
  __device__ int64_t operator()(int64_t w) const { return __popc(mask[w]); }
};
struct TileCountF {
  const int* kept;
  __device__ int64_t operator()(int64_t t) const { return kept[t]; }
};

// Column numbers of a thread's entries of a tile: four of each quarter (past the end: -1).
__device__ inline void kept_load(const int32_t* __restrict__ colind, int64_t tile0, int64_t nnz, int4 (&c)[4]) {
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int64_t e = tile0 + 1024 * u + 4 * threadIdx.x;
    if (e + 3 < nnz) {
      c[u] = *reinterpret_cast<const int4*>(colind + e);
    } else {
      c[u].x = e < nnz ? colind[e] : -1;
      c[u].y = e + 1 < nnz ? colind[e + 1] : -1;
      c[u].z = e + 2 < nnz ? colind[e + 2] : -1;
      c[u].w = -1;
    }
  }
}
__device__ inline unsigned kept_flag(const uint32_t* __restrict__ mask, int c) {
  return c >= 0 ? (mask[c >> 5] >> (c & 31)) & 1u : 0u;
}
__device__ inline unsigned kept_flags(const uint32_t* __restrict__ mask, const int4& c) {
  return kept_flag(mask, c.x) | kept_flag(mask, c.y) << 1 | kept_flag(mask, c.z) << 2 | kept_flag(mask, c.w) << 3;
}
__device__ inline int32_t kept_rank(const uint32_t* __restrict__ mask, const int32_t* __restrict__ rank, int c) {
  return rank[c >> 5] + __popc(mask[c >> 5] & ((1u << (c & 31)) - 1u));
}

__global__ void __launch_bounds__(256)
    k_kept_count(const int32_t* __restrict__ colind, int64_t nnz, const uint32_t* __restrict__ mask,
                 int* __restrict__ kept) {
  __shared__ int part[4];
  int4 c[4];
  kept_load(colind, (int64_t)blockIdx.x * KEPT_TILE, nnz, c);
  int n = 0;
#pragma unroll
  for (int u = 0; u < 4; u++) n += __popc(kept_flags(mask, c[u]));
  for (int off = 32; off > 0; off >>= 1) n += __shfl_down(n, off, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) kept[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// The kept entries of a tile behind those of the tiles before, in order, under their new column numbers,
// and the new places of the row starts that lie in the tile.  (16.4 M entries with their count and scans:
// 230 us; a scan of 8-byte places for all entries, a table lookup in two passes and the move: 490 us.)
__global__ void __launch_bounds__(256)
    k_kept_move(const int32_t* __restrict__ colind, const float* __restrict__ vals, int64_t nnz,
                const uint32_t* __restrict__ mask, const int32_t* __restrict__ rank, const int64_t* __restrict__ base,
                const int64_t* __restrict__ rowptr, int64_t n_rows, int32_t* __restrict__ out_col,
                float* __restrict__ out_val, int64_t* __restrict__ out_rowptr) {
  __shared__ uint64_t wave_sum[4];
  __shared__ uint16_t before[1024];  // kept entries of the tile before a group of four
  __shared__ uint8_t flags[1024];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t tile0 = (int64_t)blockIdx.x * KEPT_TILE;
  int4 c[4];
  kept_load(colind, tile0, nnz, c);
  unsigned f[4];
  uint64_t mine = 0;  // kept entries of the four groups, 16 bits each
#pragma unroll
  for (int u = 0; u < 4; u++) {
    f[u] = kept_flags(mask, c[u]);
    mine |= (uint64_t)__popc(f[u]) << (16 * u);
  }
  uint64_t incl = mine;
  for (int off = 1; off < 64; off <<= 1) {
    const uint64_t up = __shfl_up((unsigned long long)incl, off, 64);
    if (lane >= off) incl += up;
  }
  if (lane == 63) wave_sum[wave] = incl;
  __syncthreads();
  uint64_t excl = incl - mine, total = 0;
#pragma unroll
  for (int w = 0; w < 4; w++) {
    if (w < wave) excl += wave_sum[w];
    total += wave_sum[w];
  }
  const int64_t tile_base = base[blockIdx.x];
  unsigned quarter = 0;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const unsigned pre = quarter + (unsigned)((excl >> (16 * u)) & 0xffff);
    quarter += (unsigned)((total >> (16 * u)) & 0xffff);
    before[256 * u + t] = (uint16_t)pre;
    flags[256 * u + t] = (uint8_t)f[u];
    if (!f[u]) continue;
    const int64_t e = tile0 + 1024 * u + 4 * t;
    int64_t at = tile_base + pre;
    const int col[4] = {c[u].x, c[u].y, c[u].z, c[u].w};
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (f[u] >> i & 1u) {
        out_col[at] = kept_rank(mask, rank, col[i]);
        out_val[at] = vals[e + i];
        at++;
      }
  }
  __syncthreads();
  // row starts in [tile0, tile0 + KEPT_TILE), the end of the last row (and empty rows there) with the last tile
  const bool last = blockIdx.x == gridDim.x - 1;
  int64_t a = 0, b = n_rows + 1;
  while (a < b) {
    const int64_t mid = (a + b) >> 1;
    if (rowptr[mid] < tile0) a = mid + 1;
    else b = mid;
  }
  for (int64_t i = a + t; i <= n_rows; i += 256) {
    const int64_t off = rowptr[i] - tile0;
    if (!last && off >= KEPT_TILE) break;
    if (tile0 + off >= nnz) {
      out_rowptr[i] = base[gridDim.x];
    } else {
      // group of the entry: quarter off / 1024, thread off % 1024 / 4
      const int g = (int)(off >> 10) * 256 + (int)((off & 1023) >> 2);
      out_rowptr[i] = tile_base + before[g] + __popc(flags[g] & ((1u << (off & 3)) - 1u));
    }
  }
}

__global__ void __launch_bounds__(256)
    k_kept_renumber(int32_t* __restrict__ colind, int64_t nnz, const uint32_t* __restrict__ mask,
                    const int32_t* __restrict__ rank) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nnz; e += stride)
    colind[e] = kept_rank(mask, rank, colind[e]);
}

template <bool TWO>
static int mark_columns(const int32_t* colind, int64_t nnz, int64_t n_cols, int64_t n_words, uint32_t* mask) {
  hipStream_t st = stream();
  // an equal share of the words per range, at most what LDS holds
  const int64_t most = TWO ? MARK_LDS_WORDS / 2 : MARK_LDS_WORDS;
  const int64_t ranges = ceil_div(n_words, most), words = ceil_div(n_words, ranges);
  const int64_t parts = std::max<int64_t>(1, std::min(n_cus() / ranges, ceil_div(nnz, 16 * MARK_THREADS)));
  const int64_t per_part = ceil_div(ceil_div(nnz, parts), 4) * 4;
  const size_t lds = sizeof(uint32_t) * (size_t)(TWO ? 2 * words : words);
  DN_HIP(hipFuncSetAttribute((const void*)k_mark_columns<TWO>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)(sizeof(uint32_t) * MARK_LDS_WORDS)));
  dbuf<uint32_t> marks;
  DN_TRY(marks.alloc(ranges * parts * (int64_t)(lds / sizeof(uint32_t))));
  hipLaunchKernelGGL(k_mark_columns<TWO>, dim3((unsigned)ranges, (unsigned)parts), dim3(MARK_THREADS), lds, st, colind,
                     nnz, per_part, (int)words, marks.p);
  hipLaunchKernelGGL(k_merge_marks<TWO>, dim3((unsigned)ceil_div(n_words, 256)), dim3(256), 0, st, marks.p, (int)parts,
                     (int)words, n_words, mask);
  DN_LAUNCH_CHECK();
  return 0;
}

// Reading the column numbers once per range costs 4 bytes per entry and range at several TB/s, an update of
// a counter in memory 50 ps: the same at about 100 ranges out of the memory-side cache, 60 out of
// memory.  Few entries: their counters are updated before the marks of all columns are cleared and merged.
static bool marks_pay(int64_t nnz, int64_t n_words, int min_count) {
  if (min_count != 1 && min_count != 2) return false;
  const int64_t most = min_count == 2 ? MARK_LDS_WORDS / 2 : MARK_LDS_WORDS;
  return ceil_div(n_words, most) <= 48 && nnz >= 8 * n_words;
}

int column_mask_of_counts(const int32_t* colind, int64_t nnz, int64_t n_cols, int min_count, uint32_t* mask) {
  const int64_t n_words = ceil_div(n_cols, 32);
  if (n_words == 0) return 0;
  if (marks_pay(nnz, n_words, min_count))
    return min_count == 2 ? mark_columns<true>(colind, nnz, n_cols, n_words, mask)
                          : mark_columns<false>(colind, nnz, n_cols, n_words, mask);
  dbuf<int> count;
  DN_TRY(count.alloc(n_cols));
  DN_TRY(count_columns(colind, nnz, n_cols, count));
  hipLaunchKernelGGL(k_mask_of_counts, dim3((unsigned)ceil_div(n_words, 256)), dim3(256), 0, stream(), count.p, min_count,
                     n_cols, n_words, mask);
  DN_LAUNCH_CHECK();
  return 0;
}

int column_mask_of_list(const int32_t* kept, int64_t n_kept, int64_t n_cols, uint32_t* mask) {
  const int64_t n_words = ceil_div(n_cols, 32);
  if (n_words == 0) return 0;
  hipLaunchKernelGGL(k_mask_of_list, dim3((unsigned)ceil_div(n_words, 256)), dim3(256), 0, stream(), kept, n_kept, n_words,
                     mask);
  DN_LAUNCH_CHECK();
  return 0;
}

int keep_columns(dnpeff_csr* A, const uint32_t* mask, int32_t** new_to_og) {
  hipStream_t st = stream();
  const int64_t n_words = ceil_div(A->n_cols, 32), nnz = A->nnz, tiles = ceil_div(nnz, KEPT_TILE);
  dbuf<int32_t> rank, list;
  dbuf<int> kept;
  dbuf<int64_t> base;
  DN_TRY(rank.alloc(n_words + 1));
  unsigned long long* host = nullptr;
  DN_TRY(host_words(&host));
  int64_t* totals = reinterpret_cast<int64_t*>(host);
  DN_TRY(exclusive_scan(MaskBitsF{mask}, n_words, rank.p, totals));
  DN_TRY(kept.alloc(tiles));
  DN_TRY(base.alloc(tiles + 1));
  if (tiles)
    hipLaunchKernelGGL(k_kept_count, dim3((unsigned)tiles), dim3(256), 0, st, A->colind, nnz, mask, kept.p);
  DN_LAUNCH_CHECK();
  DN_TRY(exclusive_scan(TileCountF{kept}, tiles, base.p, totals + 1));
  DN_HIP(hipStreamSynchronize(st));
  const int64_t n_cols = totals[0], n_kept = totals[1];
  if (new_to_og) {
    DN_TRY(list.alloc(n_cols));
    if (n_words)
      hipLaunchKernelGGL(k_list_of_mask, dim3((unsigned)ceil_div(n_words, 256)), dim3(256), 0, st, mask, rank.p, n_words,
                         list.p);
    DN_LAUNCH_CHECK();
  }
  if (n_kept == nnz) {
    if (nnz) {
      const int64_t g = std::min<int64_t>(ceil_div(nnz, 256), 16384);
      hipLaunchKernelGGL(k_kept_renumber, dim3((unsigned)g), dim3(256), 0, st, A->colind, nnz, mask, rank.p);
      DN_LAUNCH_CHECK();
    }
  } else {
    dbuf<int32_t> out_col;
    dbuf<float> out_val;
    dbuf<int64_t> out_rowptr;
    DN_TRY(out_col.alloc(n_kept));
    DN_TRY(out_val.alloc(n_kept));
    DN_TRY(out_rowptr.alloc(A->n_rows + 1));
    hipLaunchKernelGGL(k_kept_move, dim3((unsigned)tiles), dim3(256), 0, st, A->colind, A->vals, nnz, mask, rank.p, base.p,
                       A->rowptr, A->n_rows, out_col.p, out_val.p, out_rowptr.p);
    DN_LAUNCH_CHECK();
    dfree(A->colind);
    dfree(A->vals);
    dfree(A->rowptr);
    A->colind = out_col.release();
    A->vals = out_val.release();
    A->rowptr = out_rowptr.release();
    A->nnz = n_kept;
  }
  if (new_to_og) *new_to_og = list.release();
  A->n_cols = n_cols;
  return 0;
}

}  // namespace dn
