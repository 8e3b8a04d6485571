// CSR loader on the device: upload, row normalisation, column compaction,
// column retention, transposed CSR, ||A||^2.  Integer results are bit-exact
// with the reference's host code; see include/dnpeff.h for the citations.
#include "dnpeff_internal.hpp"
#include "host_parts.hpp"
#include "scan.hpp"

#include <cmath>
#include <cstdlib>

#include <algorithm>
#include <cctype>
#include <cstdarg>
#include <cstring>
#include <memory>
#include <new>
#include <vector>

namespace dn {

// ---------------------------------------------------------------------------
// Library state
// ---------------------------------------------------------------------------
static thread_local char g_error[1024] = "";
static hipStream_t g_stream = nullptr;
static int g_n_cus = 0;

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}
void clear_error() { g_error[0] = 0; }

static hipStream_t g_side_stream = nullptr;
static bool g_on_side_stream = false;
static hipEvent_t g_side_done = nullptr;  // recorded on the side stream; nullptr = nothing pending

hipStream_t stream() {
  if (g_on_side_stream) return g_side_stream;
  if (!g_stream) {
    if (hipStreamCreate(&g_stream) != hipSuccess) {
      fprintf(stderr, "dnpeff: hipStreamCreate failed (no usable GPU?)\n");
      abort();
    }
  }
  return g_stream;
}

// Work launched between side_stream_begin() and side_stream_end() goes to a second stream of the
// same (default) priority: it starts once everything launched so far on the library stream has
// finished, and runs beside what the library stream gets afterwards, until side_stream_join()
// makes the library stream wait for it.
int side_stream_begin() {
  if (!g_side_stream) DN_HIP(hipStreamCreate(&g_side_stream));
  static hipEvent_t fork = nullptr;
  if (!fork) DN_HIP(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
  DN_HIP(hipEventRecord(fork, stream()));
  DN_HIP(hipStreamWaitEvent(g_side_stream, fork, 0));
  g_on_side_stream = true;
  return 0;
}
int side_stream_end() {
  static hipEvent_t done = nullptr;
  if (!done) DN_HIP(hipEventCreateWithFlags(&done, hipEventDisableTiming));
  g_on_side_stream = false;
  DN_HIP(hipEventRecord(done, g_side_stream));
  g_side_done = done;
  return 0;
}
int side_stream_join() {
  if (!g_side_done) return 0;
  hipEvent_t e = g_side_done;
  g_side_done = nullptr;
  DN_HIP(hipStreamWaitEvent(stream(), e, 0));
  return 0;
}

// The two streams by themselves, and where stream() points, for callers that order work between
// them with events of their own.
hipStream_t side_stream_handle() {
  if (!g_side_stream && hipStreamCreate(&g_side_stream) != hipSuccess) return nullptr;
  return g_side_stream;
}
void side_stream_route(bool on) { g_on_side_stream = on && g_side_stream != nullptr; }
bool side_stream_routed() { return g_on_side_stream; }
bool side_stream_pending() { return g_side_done != nullptr; }

int n_cus() {
  if (!g_n_cus) {
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, 0) == hipSuccess) g_n_cus = p.multiProcessorCount;
    if (g_n_cus <= 0) g_n_cus = 256;
  }
  return g_n_cus;
}

struct tuning_entry {
  const char* name;
  double tuning_t::*field;
};
static const tuning_entry g_tuning_table[] = {
    {"dense_fill", &tuning_t::dense_fill},       {"panels", &tuning_t::panels},
    {"sweep_bytes", &tuning_t::sweep_bytes},     {"sweep_min", &tuning_t::sweep_min},
    {"sweep_waves", &tuning_t::sweep_waves},     {"sweep_lag", &tuning_t::sweep_lag},
    {"sweep_spin", &tuning_t::sweep_spin},       {"spmm_t_slices", &tuning_t::spmm_t_slices},
    {"split_bf16", &tuning_t::split_bf16},       {"fused_gram", &tuning_t::fused_gram},
    {"h_tile_mb", &tuning_t::h_tile_mb},         {"tiled_h", &tuning_t::tiled_h},
    {"topk_fast_cap", &tuning_t::topk_fast_cap}, {"verbose", &tuning_t::verbose},
    {"n_lists", &tuning_t::n_lists},             {"t_lists", &tuning_t::t_lists},
    {"nl_piece_cols", &tuning_t::nl_piece_cols}, {"nl_lag", &tuning_t::nl_lag},
    {"nl_extra_mb", &tuning_t::nl_extra_mb},
    {"nl_spin", &tuning_t::nl_spin},             {"nl_wgs", &tuning_t::nl_wgs},
    {"gram_beside", &tuning_t::gram_beside},
    {"gram_fold", &tuning_t::gram_fold},         {"xg_wgs", &tuning_t::xg_wgs},
    {"h_overlap", &tuning_t::h_overlap},         {"pad_rank", &tuning_t::pad_rank},
};

static tuning_t tuning_from_env() {
  tuning_t t;
  for (const tuning_entry& e : g_tuning_table) {
    char var[64] = "DNPEFF_";
    size_t k = strlen(var);
    for (const char* c = e.name; *c && k + 1 < sizeof(var); c++) var[k++] = (char)toupper((unsigned char)*c);
    var[k] = 0;
    if (const char* v = getenv(var)) t.*(e.field) = atof(v);
  }
  return t;
}

tuning_t& tuning() {
  static tuning_t t = tuning_from_env();
  return t;
}

// ids[b] = XCD that workgroup b of the probe runs on (hardware register XCC_ID, bits 3:0)
__global__ void k_xcd_probe(int* ids) {
  if (threadIdx.x == 0) ids[blockIdx.x] = __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)) & 15;
}

// The kernels that pin work to an XCD (swept pieces of A H^T, component slices of A^T W) count on
// the dispatcher dealing the workgroups of a launch to SWEEP_XCDS XCDs round-robin by their
// number: workgroups b, b + 8, b + 16, ... on one XCD, the eight classes on eight different ones
// (which XCD a class gets does not matter).  Checked once per process with a probe launch; where
// it does not hold (another partition mode, another part) those plans are not made: plain
// panels, one slice.
bool xcd_round_robin() {
  static int state = -1;
  if (state >= 0) return state == 1;
  state = 0;
  constexpr int N = 64 * SWEEP_XCDS;
  int* ids = nullptr;
  if (dmalloc(&ids, N)) return false;
  int h[N];
  hipLaunchKernelGGL(k_xcd_probe, dim3(N), dim3(64), 0, stream(), ids);
  if (hipGetLastError() == hipSuccess &&
      copy_down(h, ids, sizeof(int) * N) == hipSuccess) {
    bool ok = true;
    unsigned seen = 0;
    for (int x = 0; x < SWEEP_XCDS; x++) {
      for (int b = x; b < N; b += SWEEP_XCDS) ok = ok && h[b] == h[x];
      ok = ok && !(seen & (1u << h[x]));
      seen |= 1u << h[x];
    }
    state = ok ? 1 : 0;
  }
  dfree(ids);
  clear_error();
  if (state == 0 && tuning().verbose != 0.0)
    fprintf(stderr, "dnpeff: workgroups are not dealt to %d XCDs round-robin: no swept pieces, no "
                    "component slices\n", SWEEP_XCDS);
  return state == 1;
}

struct KeepMaskF {
  const int* count;
  int min_count;
  __device__ int64_t operator()(int64_t i) const { return count[i] >= min_count ? 1 : 0; }
};
struct CountsF {
  const int* count;
  __device__ int64_t operator()(int64_t i) const { return count[i]; }
};
struct KeptEntryF {
  const int32_t* colind;
  const int32_t* table;
  __device__ int64_t operator()(int64_t e) const { return table[colind[e]] != -1 ? 1 : 0; }
};
struct RowChunksF {
  const int64_t* rowptr;
  int64_t chunk;
  __device__ int64_t operator()(int64_t i) const {
    int64_t len = rowptr[i + 1] - rowptr[i];
    return (len + chunk - 1) / chunk;
  }
};
struct LongColF {
  const int64_t* colptr;
  int64_t limit;
  __device__ int64_t operator()(int64_t j) const {
    return (colptr[j + 1] - colptr[j]) > limit ? 1 : 0;
  }
};

int scan_keep_mask(const int* count, int min_count, int64_t n, int32_t* out) {
  return exclusive_scan(KeepMaskF{count, min_count}, n, out);
}
int scan_counts_i64(const int* count, int64_t n, int64_t* out, int64_t* total) {
  return exclusive_scan(CountsF{count}, n, out, total);
}
int scan_kept_entries(const int32_t* colind, const int32_t* table, int64_t nnz, int64_t* out) {
  return exclusive_scan(KeptEntryF{colind, table}, nnz, out);
}
int scan_row_chunks(const int64_t* rowptr, int64_t chunk, int64_t n, int64_t* out, int64_t* total) {
  return exclusive_scan(RowChunksF{rowptr, chunk}, n, out, total);
}
int scan_long_cols(const int64_t* colptr, int64_t limit, int64_t n, int32_t* out, int64_t* total) {
  return exclusive_scan(LongColF{colptr, limit}, n, out, total);
}

// ---------------------------------------------------------------------------
// Loader kernels
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(256) k_pef_rowptr(int64_t n_rows, int64_t k, int64_t* rowptr) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i <= n_rows; i += stride)
    rowptr[i] = i * k;
}

// vals[e] /= (norms[row] + eps); one workgroup walks one row at a time.
__global__ void __launch_bounds__(256) k_normalize_rows(const int64_t* __restrict__ rowptr,
                                                        float* __restrict__ vals,
                                                        const float* __restrict__ norms, float eps,
                                                        int64_t n_rows) {
  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    const float d = norms[row] + eps;
    const int64_t e1 = rowptr[row + 1];
    for (int64_t e = rowptr[row] + threadIdx.x; e < e1; e += 256) vals[e] = vals[e] / d;
  }
}

__global__ void __launch_bounds__(256)
    k_col_hist(const int32_t* __restrict__ colind, int64_t nnz, int* __restrict__ count) {
  int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nnz; e += stride)
    atomicAdd(&count[colind[e]], 1);
}

// og_to_new[i] = pos[i] if kept else -1; new_to_og[pos[i]] = i.
__global__ void __launch_bounds__(256)
    k_build_maps(const int* __restrict__ count, int min_count, const int32_t* __restrict__ pos,
                 int64_t n_cols, int32_t* __restrict__ og_to_new, int32_t* __restrict__ new_to_og) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_cols; i += stride) {
    if (count[i] >= min_count) {
      og_to_new[i] = pos[i];
      new_to_og[pos[i]] = (int32_t)i;
    } else {
      og_to_new[i] = -1;
    }
  }
}

// table[c] = -1 for the columns of the head, c for the others
__global__ void __launch_bounds__(256)
    k_tail_table(const int32_t* __restrict__ og_to_new, int64_t n_cols, int32_t* __restrict__ table) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_cols; i += stride)
    table[i] = og_to_new[i] >= 0 ? -1 : (int32_t)i;
}

// Entries of the head's columns into the dense block; a workgroup per row.  Every element must
// receive one addition: an addition that finds something other than zero in its element means
// that the row holds the column twice (*repeats counts them; a repeat whose earlier values were
// all exactly zero goes unnoticed and changes nothing: 0 + x has one value whatever the order).
__global__ void __launch_bounds__(256)
    k_head_fill(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind,
                const float* __restrict__ vals, int64_t n_rows, const int32_t* __restrict__ slot_of,
                float* __restrict__ cm, int64_t n_pad, int* __restrict__ repeats) {
  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    const int64_t e1 = rowptr[row + 1];
    for (int64_t e = rowptr[row] + threadIdx.x; e < e1; e += 256) {
      const int32_t k = slot_of[colind[e]];
      if (k >= 0 && atomicAdd(&cm[(int64_t)k * n_pad + row], vals[e]) != 0.0f) atomicAdd(repeats, 1);
    }
  }
}

// bounds[p] = first column c with colptr[c] >= p * nnz / P  (bounds[0] = 0, bounds[P] = n_cols):
// P panels of consecutive columns with about the same number of entries each.
__global__ void __launch_bounds__(256)
    k_panel_bounds(const int64_t* __restrict__ colptr, int64_t n_cols, int64_t nnz, int P,
                   int32_t* __restrict__ bounds) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p > P) return;
  if (p == 0) { bounds[0] = 0; return; }
  if (p == P) { bounds[P] = (int32_t)n_cols; return; }
  const int64_t target = (int64_t)(((__int128)nnz * p) / P);
  int64_t lo = 0, hi = n_cols;  // smallest c in [0, n_cols] with colptr[c] >= target
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (colptr[mid] >= target) hi = mid; else lo = mid + 1;
  }
  bounds[p] = (int32_t)lo;
}

// Regroups the entries of each row by column panel, keeping their order inside a panel (a
// stable split, so the result does not depend on how the hardware schedules the lanes), and
// records where each (row, panel) segment starts.  One workgroup per row at a time: a counting
// pass, a scan over the panels, then tiles of 256 entries in order; within a tile an entry's
// rank among the entries of its panel comes from wave ballots over the bits of the panel
// number plus the per-wave counts of the earlier waves.
constexpr int MAX_PANELS = 3072;

__global__ void __launch_bounds__(256)
    k_panel_split(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind,
                  const float* __restrict__ vals, int64_t n_rows, int P, int bits,
                  const int32_t* __restrict__ bounds, int64_t* __restrict__ seg,
                  int32_t* __restrict__ pcol, float* __restrict__ pval,
                  const int64_t* __restrict__ out_begin) {
  // out_begin (or NULL): the panels end below the matrix's last column; row i's entries below
  // bounds[P] (out_begin[i + 1] - out_begin[i] of them, anywhere in the row) go to
  // out_begin[i] .. of pcol / pval, and the segment offsets count from there; the others are left
  // out
  __shared__ int32_t bnd[MAX_PANELS + 1];
  __shared__ int hist[MAX_PANELS];
  __shared__ int cursor[MAX_PANELS];         // next free position of each panel, relative to e0
  __shared__ uint8_t wcnt[4][MAX_PANELS];    // entries of a panel in one wave of a tile (<= 64)
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int i = tid; i <= P; i += 256) bnd[i] = bounds[i];
  auto panel_of = [&](int32_t col) {
    int lo = 0, hi = P;  // largest p < P with bnd[p] <= col
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (bnd[mid] <= col) lo = mid; else hi = mid;
    }
    return lo;
  };
  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    const int64_t e0 = rowptr[row], e1 = rowptr[row + 1];
    const int64_t o0 = out_begin ? out_begin[row] : e0;
    const int64_t o1 = out_begin ? out_begin[row + 1] : e1;
    const int32_t col_end = bounds[P];
    __syncthreads();
    for (int i = tid; i < P; i += 256) {
      hist[i] = 0;
      wcnt[0][i] = wcnt[1][i] = wcnt[2][i] = wcnt[3][i] = 0;
    }
    __syncthreads();
    for (int64_t e = e0 + tid; e < e1; e += 256)
      if (colind[e] < col_end) atomicAdd(&hist[panel_of(colind[e])], 1);
    __syncthreads();
    // exclusive scan of the panel counts: each thread sums a run of consecutive panels, the
    // run totals are scanned by thread 0
    {
      const int per = (P + 255) / 256, p0 = tid * per;
      int s = 0;
      for (int q = p0; q < p0 + per && q < P; q++) s += hist[q];
      __syncthreads();
      if (p0 < P) cursor[p0] = s;  // run total, parked in the run's first slot
      __syncthreads();
      if (tid == 0) {
        int run = 0;
        for (int q = 0; q < P; q += per) {
          const int t = cursor[q];
          cursor[q] = run;
          run += t;
        }
      }
      __syncthreads();
      if (p0 < P) {
        int run = cursor[p0];
        for (int q = p0; q < p0 + per && q < P; q++) {
          cursor[q] = run;
          seg[row * (P + 1) + q] = o0 + run;
          run += hist[q];
        }
      }
    }
    if (tid == 0) seg[row * (P + 1) + P] = o1;
    __syncthreads();
    for (int64_t base = e0; base < e1; base += 256) {
      const int64_t e = base + tid;
      bool active = e < e1;
      int32_t col = 0;
      float v = 0.0f;
      int pid = 0;
      if (active) {
        col = colind[e];
        active = col < col_end;
      }
      if (active) {
        v = vals[e];
        pid = panel_of(col);
      }
      unsigned long long mask = __ballot(active);
      for (int b = 0; b < bits; b++) {
        const bool bit = (pid >> b) & 1;
        const unsigned long long bal = __ballot(active && bit);
        mask &= bit ? bal : ~bal;
      }
      const int rank = __popcll(mask & ((1ull << lane) - 1ull));
      if (active && rank == 0) wcnt[wave][pid] = (uint8_t)__popcll(mask);
      __syncthreads();
      int off = 0, tot = 0;
      if (active) {
        for (int w = 0; w < 4; w++) {
          const int c = wcnt[w][pid];
          if (w < wave) off += c;
          tot += c;
        }
        const int64_t pos = o0 + cursor[pid] + off + rank;
        pcol[pos] = col;
        pval[pos] = v;
      }
      __syncthreads();
      // the last entry of each panel in the tile (last wave that holds it, last lane of its
      // mask) moves the panel's cursor on and clears its counts
      if (active) {
        bool last_wave = true;
        for (int w = wave + 1; w < 4; w++) last_wave = last_wave && wcnt[w][pid] == 0;
        if (last_wave && rank == __popcll(mask) - 1) cursor[pid] += tot;
      }
      __syncthreads();
      if (active && rank == 0) wcnt[wave][pid] = 0;
    }
  }
}

// ---------------------------------------------------------------------------
// Threshold compaction: (i, x[i] / divisor) of the elements with x[i] / divisor >= threshold, in
// ascending order.  A workgroup owns a run of whole tiles of THR_TILE elements; one launch counts
// what passes per run, the next adds up the counts of the runs before its own and writes.  The
// second read of x comes from the memory-side cache at the sizes of a component (24 MB at 6 M
// columns), and no per-element positions are kept: 40 us per 6 M elements for both launches, where
// a scan of positions (8 bytes per element written and read) took 78.  A thread takes four consecutive
// elements, so a tile's order is lane order inside wave order: ranks from a shuffle prefix sum
// and the counts of the earlier waves.
// ---------------------------------------------------------------------------
constexpr int THR_TILE = 1024;      // elements of a workgroup step: 256 threads x 4
constexpr int THR_MAX_WGS = 1024;   // runs (their counts are added up by every workgroup)

// one tile: the four quotients of a thread (x past the end of the array fails the test)
template <bool VEC4>
__device__ inline void thr_load(const float* __restrict__ x, int64_t i, int64_t n, float divisor,
                                float (&v)[4], bool (&ok)[4], float threshold) {
  if (VEC4 && i + 3 < n) {
    const float4 t = *reinterpret_cast<const float4*>(x + i);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      v[k] = v[k] / divisor;
      ok[k] = v[k] >= threshold;
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const bool in = i + k < n;
      v[k] = (in ? x[i + k] : 0.0f) / divisor;
      ok[k] = in && v[k] >= threshold;
    }
  }
}

template <bool VEC4>
__global__ void __launch_bounds__(256)
    k_threshold_count(const float* __restrict__ x, float divisor, float threshold, int64_t n, int64_t per_wg,
                      int* __restrict__ counts) {
  const int64_t e0 = (int64_t)blockIdx.x * per_wg, e1 = e0 + per_wg < n ? e0 + per_wg : n;
  int c = 0;
  for (int64_t b = e0 + 4 * (int)threadIdx.x; b < e1; b += THR_TILE) {
    float v[4];
    bool ok[4];
    thr_load<VEC4>(x, b, n, divisor, v, ok, threshold);
    c += (int)ok[0] + (int)ok[1] + (int)ok[2] + (int)ok[3];
  }
  __shared__ int sh[4];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

template <bool VEC4>
__global__ void __launch_bounds__(256)
    k_threshold_write(const float* __restrict__ x, float divisor, float threshold, int64_t n, int64_t per_wg,
                      const int* __restrict__ counts, int32_t* __restrict__ idx_out,
                      float* __restrict__ val_out, unsigned long long* __restrict__ total) {
  __shared__ int64_t sh_base[4];
  __shared__ int wcnt[2][4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int64_t base = 0;
  for (int q = threadIdx.x; q < (int)blockIdx.x; q += 256) base += counts[q];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) base += __shfl_xor(base, off);
  if (lane == 0) sh_base[wave] = base;
  __syncthreads();
  base = sh_base[0] + sh_base[1] + sh_base[2] + sh_base[3];
  if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0)
    *total = (unsigned long long)(base + counts[blockIdx.x]);
  if (counts[blockIdx.x] == 0) return;  // (the whole workgroup)
  const int64_t e0 = (int64_t)blockIdx.x * per_wg, e1 = e0 + per_wg < n ? e0 + per_wg : n;
  int it = 0;
  for (int64_t t0 = e0; t0 < e1; t0 += THR_TILE, it++) {
    const int64_t i = t0 + 4 * (int)threadIdx.x;
    float v[4];
    bool ok[4];
    thr_load<VEC4>(x, i, n, divisor, v, ok, threshold);
    const int c = (int)ok[0] + (int)ok[1] + (int)ok[2] + (int)ok[3];
    int incl = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off);
      if (lane >= off) incl += up;
    }
    if (lane == 63) wcnt[it & 1][wave] = incl;
    __syncthreads();  // (the other set of counts is written next: one barrier per tile)
    int before = incl - c, all = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const int t = wcnt[it & 1][w];
      if (w < wave) before += t;
      all += t;
    }
    int64_t at = base + before;
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (ok[k]) {
        idx_out[at] = (int32_t)(i + k);
        val_out[at] = v[k];
        at++;
      }
    base += all;
  }
}

// The same for a caller on the host: x is read once.  A workgroup notes its first THR_KEEP finds (x itself), in order,
// and counts all; k_threshold_pack divides and puts the notes side by side into a pinned buffer where that holds them
// all.  6 M elements, 60,000 kept: 6.6 and 13.2 us; counting, writing and gathering took 6.7, 10.6 and 11.6 and a wait
// in between.  Bound by its instructions and the read of x: BY_CUT compares x with the least x whose quotient passes
// (threshold_cut; dividing every x: 8.7 us); two tiles are asked for at once, one barrier for the two (one: 7.2 us,
// four: 7.9).
constexpr int THR_KEEP = 1024;  // notes per workgroup: 8 KB of LDS, 8 MB on the device
constexpr int THR_STEP = 2;     // tiles per step
constexpr unsigned long long THR_FITS = 1ull << 40;

template <bool VEC4, bool BY_CUT>
__global__ void __launch_bounds__(256)
    k_threshold_find(const float* __restrict__ x, float divisor, float threshold, int64_t n, int64_t per_wg,
                     int* __restrict__ counts, uint2* __restrict__ found) {
  __shared__ uint2 note[THR_KEEP];
  __shared__ int wcnt[2][THR_STEP][4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t e0 = (int64_t)blockIdx.x * per_wg, e1 = e0 + per_wg < n ? e0 + per_wg : n;
  int base = 0, it = 0;
  for (int64_t t0 = e0; t0 < e1; t0 += THR_STEP * THR_TILE, it ^= 1) {
    const int64_t i0 = t0 + 4 * (int)threadIdx.x;
    float v[THR_STEP][4];  // past the end: NaN, which no test passes
    if (VEC4 && (e1 - t0 >= THR_STEP * THR_TILE || (e1 - t0) % THR_TILE == 0)) {
#pragma unroll
      for (int u = 0; u < THR_STEP; u++) {
        float4 q{NAN, NAN, NAN, NAN};
        if (t0 + u * THR_TILE < e1) q = *reinterpret_cast<const float4*>(x + i0 + u * THR_TILE);
        v[u][0] = q.x; v[u][1] = q.y; v[u][2] = q.z; v[u][3] = q.w;
      }
    } else {
#pragma unroll
      for (int u = 0; u < THR_STEP; u++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int64_t i = i0 + u * THR_TILE + k;
          v[u][k] = i < e1 ? x[i] : NAN;
        }
    }
    bool ok[THR_STEP][4];
    int before[THR_STEP];
#pragma unroll
    for (int u = 0; u < THR_STEP; u++) {
      int low = 0, all = 0;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        ok[u][k] = (BY_CUT ? v[u][k] : v[u][k] / divisor) >= threshold;
        const uint64_t b = __ballot(ok[u][k]);
        low = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, low));
        all += __popcll(b);
      }
      before[u] = low;
      if (lane == 0) wcnt[it][u][wave] = all;
    }
    __syncthreads();  // (the other set of counts is written next)
#pragma unroll
    for (int u = 0; u < THR_STEP; u++) {
      int at = base + before[u];
#pragma unroll
      for (int w = 0; w < 4; w++) {
        const int c = wcnt[it][u][w];
        if (w < wave) at += c;
        base += c;
      }
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (ok[u][k]) {
          if (at < THR_KEEP) note[at] = uint2{(uint32_t)(i0 + u * THR_TILE + k), __float_as_uint(v[u][k])};
          at++;
        }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = base;
  const int noted = base < THR_KEEP ? base : THR_KEEP;
  for (int i = threadIdx.x; i < noted; i += 256) found[(int64_t)blockIdx.x * THR_KEEP + i] = note[i];
}

// word (pinned; the host waits for it, not for the kernel): the number of finds and, in THR_FITS, whether idx and val (room
// for `room` of them, a multiple of 4) will hold them.  Every workgroup
// adds up the counts for itself; a thread looks its four finds up in the sums, so that whole lines go over the link.
__global__ void __launch_bounds__(256)
    k_threshold_pack(const int* __restrict__ counts, int n_runs, const uint2* __restrict__ found, float divisor, int room,
                     int4* __restrict__ idx, float4* __restrict__ val, unsigned long long* __restrict__ word) {
  static_assert(THR_MAX_WGS == 4 * 256, "a thread adds up four runs");
  __shared__ int start[THR_MAX_WGS + 1];
  __shared__ int wsum[4], crowded[4];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  int c[4], sum = 0, most = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    c[k] = 4 * t + k < n_runs ? counts[4 * t + k] : 0;
    sum += c[k];
    most = max(most, c[k]);
  }
  int incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int up = __shfl_up(incl, off);
    if (lane >= off) incl += up;
  }
  const bool over = __any(most > THR_KEEP);
  if (lane == 63) {
    wsum[wave] = incl;
    crowded[wave] = over;
  }
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wave; w++) run += wsum[w];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    start[4 * t + k] = run;
    run += c[k];
  }
  if (t == 255) start[THR_MAX_WGS] = run;
  __syncthreads();
  const int total = start[THR_MAX_WGS];
  const bool fits = total <= room && !(crowded[0] | crowded[1] | crowded[2] | crowded[3]);
  if (blockIdx.x == 0 && t == 0)
    __hip_atomic_store(word, (unsigned long long)total | (fits ? THR_FITS : 0ull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (!fits) return;
  for (int q = blockIdx.x * 256 + t; 4 * q < total; q += gridDim.x * 256) {
    int g = 0;  // the last run that starts at or before the first of the four
#pragma unroll
    for (int half = THR_MAX_WGS / 2; half > 0; half >>= 1)
      if (start[g + half] <= 4 * q) g += half;
    uint2 f[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int o = 4 * q + k;
      f[k] = uint2{0u, 0u};
      if (o < total) {
        while (o >= start[g + 1]) g++;
        f[k] = found[(int64_t)g * THR_KEEP + (o - start[g])];
      }
    }
    idx[q] = int4{(int)f[0].x, (int)f[1].x, (int)f[2].x, (int)f[3].x};
    val[q] = float4{__uint_as_float(f[0].y) / divisor, __uint_as_float(f[1].y) / divisor, __uint_as_float(f[2].y) / divisor,
                    __uint_as_float(f[3].y) / divisor};
  }
}

__global__ void __launch_bounds__(256) k_fill_i32(int32_t* p, int64_t n, int32_t v) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) p[i] = v;
}

// old_to_new[kept[i]] = i; for a column listed twice the last position wins,
// as in the reference's sequential loop.
__global__ void __launch_bounds__(256)
    k_retain_table(const int32_t* __restrict__ kept, int64_t n_kept, int32_t* __restrict__ table) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_kept; i += stride)
    atomicMax(&table[kept[i]], (int32_t)i);
}

__global__ void __launch_bounds__(256)
    k_remap_cols(int32_t* __restrict__ colind, int64_t nnz, const int32_t* __restrict__ table) {
  int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nnz; e += stride)
    colind[e] = table[colind[e]];
}

// Order-preserving removal of entries whose column was dropped.
__global__ void __launch_bounds__(256)
    k_compact_entries(const int32_t* __restrict__ colind, const float* __restrict__ vals,
                      int64_t nnz, const int32_t* __restrict__ table,
                      const int64_t* __restrict__ newpos, int32_t* __restrict__ out_col,
                      float* __restrict__ out_val) {
  int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nnz; e += stride) {
    int32_t c = table[colind[e]];
    if (c != -1) {
      int64_t p = newpos[e];
      out_col[p] = c;
      out_val[p] = vals[e];
    }
  }
}

__global__ void __launch_bounds__(256)
    k_remap_rowptr(int64_t* __restrict__ rowptr, int64_t n_rows, const int64_t* __restrict__ newpos) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i <= n_rows; i += stride)
    rowptr[i] = newpos[rowptr[i]];
}

// One row of the stable transposition: entry e of this row goes to the next
// free slot of its column.  Rows are issued in ascending order on one stream
// and a row holds each column at most once, so every column ends up in
// ascending row order.
__global__ void __launch_bounds__(256)
    k_transpose_row(int32_t row, int64_t e0, int64_t e1, const int32_t* __restrict__ colind,
                    const float* __restrict__ vals, const int64_t* __restrict__ colptr,
                    int* __restrict__ cursor, int32_t* __restrict__ rowind,
                    float* __restrict__ tvals) {
  int64_t e = e0 + (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= e1) return;
  int32_t j = colind[e];
  int64_t p = colptr[j] + atomicAdd(&cursor[j], 1);
  rowind[p] = row;
  tvals[p] = vals[e];
}

// The transposed copy of rows that hold their columns in ascending order, range by range of columns: a row's entries of
// a range lie side by side.  The eight waves of a workgroup take an eighth of the rows each: they count their entries of
// the range's columns in LDS (two counters of 16 bits to a word), the counts become offsets, column by column and wave by
// wave, and every wave places its entries row after row, which is the order of the columns, into LDS, from where they go
// out in one piece.  at[range][row] = entries of the row before the range.
//
// 256 rows of 220 k entries, 22 M columns: 0.46 ms and 0.09 for the table, where the rows one by one take 8.9 (a launch and an update of a
// counter in memory per entry, and the columns counted and looked over before and after); with entries stored straight to their
// columns, 2.4: their lines leave the L2s before they are full.
constexpr int RANGE_SHIFT = 11, RANGE_COLS = 1 << RANGE_SHIFT;
constexpr int RANGE_WAVES = 8;
constexpr int RANGE_STAGED = 5376;    // entries that LDS holds beside the counters, two workgroups to a CU
constexpr int RANGE_MOST = 65535;     // entries of a range (the counters' 16 bits)
constexpr int RANGE_AHEAD = 16;       // rows whose entries are asked for at a time
constexpr size_t RANGE_LDS = 4 * (size_t)(RANGE_WAVES * RANGE_COLS / 2) + 8 * (size_t)RANGE_STAGED;

// *unfit (a pinned word) = 1 unless the first columns of every row ascend: rows in no order show it here, before room is made.
__global__ void __launch_bounds__(256)
    k_range_probe(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind, int* __restrict__ unfit) {
  const int64_t e = rowptr[blockIdx.x] + 1 + threadIdx.x;
  if (__any(e < rowptr[blockIdx.x + 1] && colind[e - 1] >= colind[e]) && (threadIdx.x & 63) == 0) *unfit = 1;
}

// (A wave that sees two columns the other way round stores nothing, and none goes on once one has: the gaps between columns in
// no order add up to far more than the table.)
__global__ void __launch_bounds__(256)
    k_range_starts(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind, int64_t n, int64_t ranges,
                   uint32_t* __restrict__ at, int* uneven) {
  const int64_t row = blockIdx.x, r0 = rowptr[row], r1 = rowptr[row + 1], step = 256 * (int64_t)gridDim.y;
  for (int64_t e64 = r0 + 256 * (int64_t)blockIdx.y + (threadIdx.x & ~63); e64 <= r1; e64 += step) {  // (r1: what ends the row)
    if (__hip_atomic_load(uneven, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    const int64_t e = e64 + (threadIdx.x & 63);
    const bool in = e <= r1;
    const int32_t before = in && e > r0 ? colind[e - 1] : -1, col = e < r1 ? colind[e] : 0;
    if (__any(in && e > r0 && e < r1 && before >= col)) {
      if ((threadIdx.x & 63) == 0) __hip_atomic_store(uneven, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    if (!in) continue;
    const int64_t q0 = e > r0 ? (before >> RANGE_SHIFT) + 1 : 0, q1 = e < r1 ? col >> RANGE_SHIFT : ranges;
    for (int64_t q = q0; q <= q1; q++) at[q * n + row] = (uint32_t)(e - r0);
  }
}

// Entries of every range; *unfit (a pinned word) = 1 where there are more than RANGE_MOST, or the rows do not ascend.
__global__ void __launch_bounds__(256)
    k_range_counts(const uint32_t* __restrict__ at, int64_t n, int* __restrict__ count, const int* __restrict__ uneven,
                   int* __restrict__ unfit) {
  __shared__ int red[256];
  const uint32_t* a = at + (int64_t)blockIdx.x * n;
  int s = 0;
  for (int64_t i = threadIdx.x; i < n; i += 256) s += (int)(a[n + i] - a[i]);
  red[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    count[blockIdx.x] = red[0];
    if (red[0] > RANGE_MOST || red[0] < 0 || *uneven) *unfit = 1;
  }
}

__global__ void __launch_bounds__(64 * RANGE_WAVES)
    k_range_transpose(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind, const float* __restrict__ vals,
                      int64_t n, int64_t m, const uint32_t* __restrict__ at, const int64_t* __restrict__ base,
                      int64_t* __restrict__ colptr, int32_t* __restrict__ rowind, float* __restrict__ tvals) {
  extern __shared__ unsigned lds[];
  __shared__ int part[RANGE_WAVES];
  constexpr int WORDS = RANGE_COLS / 2;
  int* stage_row = reinterpret_cast<int*>(lds + RANGE_WAVES * WORDS);
  float* stage_val = reinterpret_cast<float*>(stage_row + RANGE_STAGED);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t range = blockIdx.x, c0 = range << RANGE_SHIFT, first = base[range];
  const int total = (int)(base[range + 1] - first);
  const bool staged = total <= RANGE_STAGED;
  unsigned* mine = lds + wave * WORDS;  // of the wave: entries of the columns, then their next places
  const int64_t per = (n + RANGE_WAVES - 1) / RANGE_WAVES, n0 = wave * per, n1 = n0 + per < n ? n0 + per : n;
  for (int x = tid; x < RANGE_WAVES * WORDS; x += 64 * RANGE_WAVES) lds[x] = 0u;
  __syncthreads();
  auto word = [&](int c) { return mine + (c >> 1); };
  auto one = [&](int c) { return 1u << (16 * (c & 1)); };
  // Entries of the wave's rows in order, up to 64 of a row at a time: take(column, whether there is one in the lane) gives
  // a place, put(row, place, value, ...) comes any time after it.
  auto sweep = [&](auto with_vals, auto take, auto put) {
    for (int64_t row0 = n0; row0 < n1; row0 += 64) {
      const int64_t own = row0 + lane < n1 ? row0 + lane : n1 - 1;
      const uint32_t* a = at + range * n + own;
      const int64_t from = rowptr[own] + a[0];
      const int len = row0 + lane < n1 ? (int)(a[n] - a[0]) : 0;
      const int rows = n1 - row0 < 64 ? (int)(n1 - row0) : 64;
      for (int r = 0; r < rows; r += RANGE_AHEAD) {
        int64_t e0[RANGE_AHEAD];
        int k[RANGE_AHEAD], col[RANGE_AHEAD], p[RANGE_AHEAD], most = 0;
        float v[RANGE_AHEAD];
#pragma unroll
        for (int u = 0; u < RANGE_AHEAD; u++) {
          const int l = r + u < 64 ? r + u : 63;
          const unsigned lo = __builtin_amdgcn_readlane((int)from, l), hi = __builtin_amdgcn_readlane((int)(from >> 32), l);
          e0[u] = (int64_t)((uint64_t)hi << 32 | lo);
          k[u] = r + u < rows ? __builtin_amdgcn_readlane(len, l) : 0;
          most = most > k[u] ? most : k[u];
          const bool in = lane < k[u];
          col[u] = in ? colind[e0[u] + lane] : 0;
          v[u] = decltype(with_vals)::value && in ? vals[e0[u] + lane] : 0.0f;
        }
        if (most <= 64) {  // (all rows' places under way at once)
#pragma unroll
          for (int u = 0; u < RANGE_AHEAD; u++) p[u] = take((int)(col[u] - c0), lane < k[u]);
#pragma unroll
          for (int u = 0; u < RANGE_AHEAD; u++) put((int32_t)(row0 + r + u), p[u], v[u], lane < k[u]);
          continue;
        }
#pragma unroll
        for (int u = 0; u < RANGE_AHEAD; u++) {
          const int32_t row = (int32_t)(row0 + r + u);
          put(row, take((int)(col[u] - c0), lane < k[u]), v[u], lane < k[u]);
          for (int b = 64; b < k[u]; b += 64) {
            const bool in = b + lane < k[u];
            const int64_t e = e0[u] + (in ? b + lane : 0);
            put(row, take((int)(colind[e] - c0), in), decltype(with_vals)::value ? vals[e] : 0.0f, in);
          }
        }
      }
    }
  };
  sweep(
      std::false_type{},
      [&](int c, bool in) {
        if (in) atomicAdd(word(c), one(c));
        return 0;
      },
      [](int32_t, int, float, bool) {});
  __syncthreads();
  // the waves' counts of a column to places: four columns to a thread
  constexpr int MINE = WORDS / (64 * RANGE_WAVES);
  static_assert(MINE * 64 * RANGE_WAVES == WORDS, "whole words to every thread");
  int entries[2 * MINE], sum = 0;
#pragma unroll
  for (int q = 0; q < MINE; q++) {
    unsigned run = 0;
    for (int w = 0; w < RANGE_WAVES; w++) {
      unsigned& x = lds[w * WORDS + MINE * tid + q];
      const unsigned k = x;
      x = run;
      run += k;  // (neither half passes 16 bits)
    }
    entries[2 * q] = (int)(run & 0xffffu);
    entries[2 * q + 1] = (int)(run >> 16);
    sum += entries[2 * q] + entries[2 * q + 1];
  }
  int incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int up = __shfl_up(incl, off);
    if (lane >= off) incl += up;
  }
  if (lane == 63) part[wave] = incl;
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wave; w++) run += part[w];
#pragma unroll
  for (int q = 0; q < MINE; q++) {
    const int c = 2 * (MINE * tid + q), next = run + entries[2 * q];
    for (int w = 0; w < RANGE_WAVES; w++) lds[w * WORDS + MINE * tid + q] += (unsigned)run | (unsigned)next << 16;
    if (c0 + c < m) colptr[c0 + c] = first + run;
    if (c0 + c + 1 < m) colptr[c0 + c + 1] = first + next;
    run = next + entries[2 * q + 1];
  }
  if (tid == 0 && range == (int64_t)gridDim.x - 1) colptr[m] = first + total;
  __syncthreads();
  sweep(
      std::true_type{},
      [&](int c, bool in) { return in ? (int)(atomicAdd(word(c), one(c)) >> (16 * (c & 1)) & 0xffffu) : 0; },  // (a row has a column once)
      [&](int32_t row, int p, float v, bool in) {
        if (!in) return;
        if (staged) {
          stage_row[p] = row;
          stage_val[p] = v;
        } else {
          rowind[first + p] = row;
          tvals[first + p] = v;
        }
      });
  if (!staged) return;
  __syncthreads();
  for (int x = tid; x < total; x += 64 * RANGE_WAVES) {
    rowind[first + x] = stage_row[x];
    tvals[first + x] = stage_val[x];
  }
}

// The transposed copy through one bit per (column, row): an entry's place in its column is the number of
// bits below its own, so all rows go at once and a column still lists its rows in order.  bits:
// [column][words].
__global__ void __launch_bounds__(256)
    k_bits_set(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind, int64_t n_rows, int words,
               uint32_t* __restrict__ bits) {
  for (int64_t row = blockIdx.y; row < n_rows; row += gridDim.y) {
    const int64_t e1 = rowptr[row + 1];
    const uint32_t bit = 1u << (row & 31);
    for (int64_t e = rowptr[row] + (int64_t)blockIdx.x * 256 + threadIdx.x; e < e1; e += (int64_t)gridDim.x * 256)
      atomicOr(&bits[(int64_t)colind[e] * words + (row >> 5)], bit);
  }
}

__global__ void __launch_bounds__(256)
    k_bits_count(const uint32_t* __restrict__ bits, int words, int64_t n_cols, int* __restrict__ count) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < n_cols; j += stride) {
    int n = 0;
    for (int w = 0; w < words; w++) n += __popc(bits[j * words + w]);
    count[j] = n;
  }
}

__global__ void __launch_bounds__(256)
    k_bits_place(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind, const float* __restrict__ vals,
                 int64_t n_rows, const uint32_t* __restrict__ bits, int words, const int64_t* __restrict__ colptr,
                 int32_t* __restrict__ rowind, float* __restrict__ tvals) {
  for (int64_t row = blockIdx.y; row < n_rows; row += gridDim.y) {
    const int64_t e1 = rowptr[row + 1];
    const uint32_t below = (1u << (row & 31)) - 1u;
    for (int64_t e = rowptr[row] + (int64_t)blockIdx.x * 256 + threadIdx.x; e < e1; e += (int64_t)gridDim.x * 256) {
      const int64_t j = colind[e];
      const uint32_t* b = bits + j * words;
      int64_t at = colptr[j] + __popc(b[row >> 5] & below);
      for (int w = 0; w < (int)(row >> 5); w++) at += __popc(b[w]);
      rowind[at] = (int32_t)row;
      tvals[at] = vals[e];
    }
  }
}

__global__ void __launch_bounds__(256)
    k_collect_long(const int64_t* __restrict__ colptr, int64_t limit, int64_t n_cols,
                   const int32_t* __restrict__ pos, int32_t* __restrict__ long_cols) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < n_cols; j += stride)
    if (colptr[j + 1] - colptr[j] > limit) long_cols[pos[j]] = (int32_t)j;
}

// Grid of a grid-stride kernel over n items (every kernel launched with it loops); a launch is
// limited to 2^32 threads in total, so grids are capped well below that.
static unsigned grid_for(int64_t n, int64_t cap = 1 << 20) {
  int64_t g = ceil_div(n, 256);
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

// sum over the columns with count >= thr of their counts (an integer sum: any order)
__global__ void __launch_bounds__(256)
    k_sum_selected(const int* __restrict__ count, int64_t n, int thr, unsigned long long* out) {
  __shared__ unsigned long long sh[256];
  unsigned long long s = 0;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    const int c = count[i];
    if (c >= thr) s += (unsigned long long)c;
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0 && sh[0]) atomicAdd(out, sh[0]);
}

// bad += 1 for every column that holds the same row twice in a row of its list (after the stable
// transposition the entries of one row of a column are adjacent)
__global__ void __launch_bounds__(256)
    k_check_repeats(const int64_t* __restrict__ colptr, const int32_t* __restrict__ rowind,
                    int64_t n_cols, int* __restrict__ bad) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < n_cols; j += stride) {
    const int64_t p1 = colptr[j + 1];
    int32_t prev = -1;
    bool rep = false;
    for (int64_t p = colptr[j]; p < p1; p++) {
      const int32_t i = rowind[p];
      rep = rep || i == prev;
      prev = i;
    }
    if (rep) atomicAdd(bad, 1);
  }
}

int count_columns(const int32_t* colind, int64_t nnz, int64_t n_cols, int* count) {
  DN_HIP(hipMemsetAsync(count, 0, sizeof(int) * (size_t)(n_cols > 0 ? n_cols : 1), stream()));
  hipLaunchKernelGGL(k_col_hist, dim3(grid_for(nnz, 65536)), dim3(256), 0, stream(), colind, nnz, count);
  DN_LAUNCH_CHECK();
  return 0;
}

// Drops entries whose table[col] == -1 and renumbers the rest (in place on A).
static int apply_column_table(dnpeff_csr* A, const int32_t* table, int64_t new_n_cols) {
  hipStream_t st = stream();
  dbuf<int64_t> newpos;
  DN_TRY(newpos.alloc(A->nnz + 1));
  DN_TRY(scan_kept_entries(A->colind, table, A->nnz, newpos));
  int64_t new_nnz = 0;
  DN_HIP(copy_down(&new_nnz, newpos + A->nnz, sizeof(int64_t)));
  if (new_nnz == A->nnz) {
    hipLaunchKernelGGL(k_remap_cols, dim3(grid_for(A->nnz)), dim3(256), 0, st, A->colind, A->nnz,
                       table);
    DN_LAUNCH_CHECK();
  } else {
    dbuf<int32_t> out_col;
    dbuf<float> out_val;
    DN_TRY(out_col.alloc(new_nnz));
    DN_TRY(out_val.alloc(new_nnz));
    hipLaunchKernelGGL(k_compact_entries, dim3(grid_for(A->nnz)), dim3(256), 0, st, A->colind,
                       A->vals, A->nnz, table, newpos.p, out_col.p, out_val.p);
    hipLaunchKernelGGL(k_remap_rowptr, dim3(grid_for(A->n_rows + 1)), dim3(256), 0, st, A->rowptr,
                       A->n_rows, newpos.p);
    DN_LAUNCH_CHECK();
    DN_HIP(hipStreamSynchronize(st));
    dfree(A->colind);
    dfree(A->vals);
    A->colind = out_col.release();
    A->vals = out_val.release();
    A->nnz = new_nnz;
  }
  DN_HIP(hipStreamSynchronize(st));
  A->n_cols = new_n_cols;
  return 0;
}

static void drop_head(dnpeff_csr* A) {
  if (A->tail) {
    dnpeff_csr_destroy(A->tail);
    A->tail = nullptr;
  }
  dfree(A->head.cols); dfree(A->head.cm); dfree(A->head.rm); dfree(A->head.ws);
  A->head = dense_head();
}

static void drop_panels(dnpeff_csr* A) {
  dfree(A->panel_bounds); A->panel_bounds = nullptr;
  dfree(A->panel_ids); A->panel_ids = nullptr;
  dfree(A->sweep_progress); A->sweep_progress = nullptr;
  dfree(A->sweep_perm); A->sweep_perm = nullptr; A->sweep_perm_key = 0;
  dfree(A->seg); A->seg = nullptr;
  dfree(A->pcol); A->pcol = nullptr;
  dfree(A->pval); A->pval = nullptr;
  dfree(A->prow); A->prow = nullptr;
  A->tail_floor = 0;
  if (A->n_panels) {  // the partial sums were sized for the panels
    dfree(A->partials); A->partials = nullptr; A->partials_floats = 0;
  }
  A->n_panels = A->n_plain = A->n_swept = 0;
  A->plan = panel_plan();
}

static void drop_slots(dnpeff_csr* A) {
  dfree(A->slots); A->slots = nullptr;
  dfree(A->spsp_at); A->spsp_at = nullptr;
  A->spsp_cuts = 0;
  A->spsp_cut = false;
}

static void drop_derived(dnpeff_csr* A) {
  A->h_lists_valid = false;
  A->tail_declined = false;
  drop_head(A);
  drop_panels(A);
  nlists_drop(A);
  tblocks_drop(A);
  fused_drop(A);
  dfree(A->colptr); A->colptr = nullptr;
  dfree(A->rowind); A->rowind = nullptr;
  dfree(A->tvals); A->tvals = nullptr;
  drop_slots(A);
  dfree(A->chunk_base); A->chunk_base = nullptr; A->n_chunks = 0;
  dfree(A->long_cols); A->long_cols = nullptr; A->n_long = 0;
  dfree(A->partials); A->partials = nullptr; A->partials_floats = 0;
}

int csr_ensure_chunks(dnpeff_csr* A) {
  if (A->chunk_base) return 0;
  DN_CHECK(A->rowptr != nullptr, "row-major copy of the matrix was released");
  DN_TRY(dmalloc(&A->chunk_base, A->n_rows + 1));
  DN_TRY(scan_row_chunks(A->rowptr, SPMM_N_CHUNK, A->n_rows, A->chunk_base));
  A->max_row_chunks = 0;
  if (A->n_rows > 0 && A->n_rows <= 4096) {
    std::vector<int64_t> base((size_t)A->n_rows + 1);
    DN_HIP(copy_down(base.data(), A->chunk_base, sizeof(int64_t) * base.size()));
    for (int64_t i = 0; i < A->n_rows; i++) A->max_row_chunks = std::max(A->max_row_chunks, base[i + 1] - base[i]);
    A->n_chunks = base[A->n_rows];
  } else {
    DN_HIP(copy_down(&A->n_chunks, A->chunk_base + A->n_rows, sizeof(int64_t)));
  }
  return 0;
}

int csr_set_panels(dnpeff_csr* S, const panel_plan& plan) {
  if (plan == S->plan) return 0;
  drop_panels(S);
  const int P0 = plan.coarse;
  if (P0 <= 0) return 0;
  DN_CHECK(P0 <= MAX_PANELS, "at most %d column panels", MAX_PANELS);
  DN_CHECK(has_row_major(S) && S->colptr, "column panels need both copies of the matrix");
  hipStream_t st = stream();
  // coarse panels: equal numbers of entries
  std::vector<int32_t> coarse((size_t)P0 + 1);
  {
    int32_t* d_coarse = nullptr;
    DN_TRY(dmalloc(&d_coarse, (int64_t)P0 + 1));
    hipLaunchKernelGGL(k_panel_bounds, dim3((unsigned)ceil_div(P0 + 1, 256)), dim3(256), 0, st,
                       S->colptr, S->n_cols, S->nnz, P0, d_coarse);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
      e = copy_down(coarse.data(), d_coarse, sizeof(int32_t) * coarse.size());
    dfree(d_coarse);
    DN_CHECK(e == hipSuccess, "building the column panels failed: %s", hipGetErrorString(e));
  }
  // A coarse panel whose part of the factor does not fit one L2 is cut into pieces that do, when
  // the rows hold entries enough per piece to be worth a segment each; those pieces are swept
  // (spmm.hip).  A raised threshold keeps the number of panels within bounds.
  std::vector<int32_t> bounds, ids, swept;
  double min_seg = plan.sweep_min;
  int P_used = P0;  // coarse panels that stay panels
  for (;;) {
    bounds.clear(); ids.clear(); swept.clear();
    const double per_coarse = (double)S->nnz / P0 / (double)(S->n_rows > 0 ? S->n_rows : 1);
    auto sweeps = [&](int c) {
      const int64_t w = (int64_t)coarse[c + 1] - coarse[c];
      return plan.sweep_cols > 0 && w > plan.sweep_cols + plan.sweep_cols / 4 &&
             per_coarse * (double)plan.sweep_cols / (double)w >= min_seg;
    };
    // The far tail: the plain panels past the last swept one.  With tail_lists their entries go
    // to slot lists and the panels end at the first of them.
    P_used = P0;
    if (plan.tail_lists) {
      int last_swept = -1;
      for (int c = 0; c < P0; c++)
        if (sweeps(c)) last_swept = c;
      if (last_swept >= 0 && last_swept + 1 < P0 && coarse[last_swept + 1] > 0) P_used = last_swept + 1;
    }
    for (int c = 0; c < P_used; c++) {
      const int64_t w = (int64_t)coarse[c + 1] - coarse[c];
      const bool sweep = sweeps(c);
      const int64_t parts = sweep ? ceil_div(w, plan.sweep_cols) : 1;
      for (int64_t q = 0; q < parts; q++) {
        (sweep ? swept : ids).push_back((int32_t)bounds.size());
        bounds.push_back((int32_t)(coarse[c] + w * q / parts));
      }
    }
    if ((int64_t)bounds.size() <= MAX_PANELS) break;
    min_seg = min_seg > 0.0 ? min_seg * 1.5 : 1.0;
  }
  const int32_t tail_floor = P_used < P0 ? coarse[P_used] : 0;
  bounds.push_back(tail_floor > 0 ? tail_floor : (int32_t)S->n_cols);
  const int P = (int)bounds.size() - 1;
  // rows' places in the panel copy when it leaves the far tail out
  int64_t nnz_panels = S->nnz;
  if (tail_floor > 0) {
    dbuf<int> below;
    int s0 = below.alloc(S->n_rows) || dmalloc(&S->prow, S->n_rows + 1) ||
             csr_rows_count_below(S, tail_floor, below.p) ||
             scan_counts_i64(below.p, S->n_rows, S->prow);
    if (!s0 && copy_down(&nnz_panels, S->prow + S->n_rows, sizeof(int64_t)) != hipSuccess) {
      set_error("building the column panels failed (row prefixes)");
      s0 = 1;
    }
    if (s0) { drop_panels(S); return 1; }
  }
  const int n_plain = (int)ids.size(), n_swept = (int)swept.size();
  ids.insert(ids.end(), swept.begin(), swept.end());

  int bits = 0;
  while ((1 << bits) < P) bits++;
  int s = dmalloc(&S->panel_bounds, (int64_t)P + 1) || dmalloc(&S->panel_ids, (int64_t)P) ||
          dmalloc(&S->sweep_progress, 256) ||
          dmalloc(&S->seg, S->n_rows * (P + 1)) || dmalloc(&S->pcol, nnz_panels + 64) ||
          dmalloc(&S->pval, nnz_panels + 64);  // (the sweep kernel reads 64 pairs at a time)
  if (!s) {
    hipError_t e = copy_up(S->panel_bounds, bounds.data(), sizeof(int32_t) * bounds.size());
    if (e == hipSuccess)
      e = copy_up(S->panel_ids, ids.data(), sizeof(int32_t) * ids.size());
    if (e == hipSuccess) {
      int64_t wgs = S->n_rows < 8192 ? S->n_rows : 8192;
      hipLaunchKernelGGL(k_panel_split, dim3((unsigned)(wgs < 1 ? 1 : wgs)), dim3(256), 0, st,
                         S->rowptr, S->colind, S->vals, S->n_rows, P, bits, S->panel_bounds, S->seg,
                         S->pcol, S->pval, (const int64_t*)S->prow);
      e = hipGetLastError();
    }
    if (e != hipSuccess) {
      set_error("building the column panels failed: %s", hipGetErrorString(e));
      s = 1;
    }
  }
  if (s) { drop_panels(S); return s; }
  S->n_panels = P;
  S->n_plain = n_plain;
  S->n_swept = n_swept;
  S->plan = plan;
  S->tail_floor = tail_floor;
  if (tuning().verbose != 0.0) {
    fprintf(stderr, "dnpeff: %d column panels: %d plain, %d cut into %d swept pieces", P_used, n_plain,
            P_used - n_plain, n_swept);
    if (tail_floor > 0)
      fprintf(stderr, "; the %d panels from column %d on (%lld entries) go to slot lists", P0 - P_used,
              (int)tail_floor, (long long)(S->nnz - nnz_panels));
    fprintf(stderr, "\n");
  }
  dfree(S->partials); S->partials = nullptr; S->partials_floats = 0;
  return 0;
}

// Panels pay when the gathered factor [n_cols, r] is far larger than the caches and there are
// rows enough to share a panel's part of it: one coarse panel per ~48 MB of the factor, 8..512
// (per ~96 MB, 8..256, at the ranks that have swept pieces), few enough for the (panel, 4
// rows) workgroups to fit one launch and for the partial sums (one [n_rows, r] block per plain
// panel) to stay within 3 GB.  On 10,000 x 65.9M,
// r = 128 (33.7 GB factor): no panels 29.3 ms, 32: 27.8, 128: 23.9, 256: 21.8, 512: 20.1 ms for
// the gathers, plus 0.1 to 0.8 ms for the sum over panels; 1024 gains 1.1 ms and loses 0.7.
// The `panels` switch overrides the number (0 = none).  Swept pieces hold `sweep_bytes` of the
// factor each (default 3 MB of the 4 MB L2 of an XCD; 0 = no sweeps) and are made where a row
// holds `sweep_min` entries per piece on average (default 4, more when there are few rows).
// Coarse panels for a sparse part of n_rows x n_cols at rank r (0 = none); `sweeps`: the rank and
// the machine have swept pieces.
int64_t coarse_panels_for(int64_t n_rows, int64_t n_cols, int r, bool sweeps) {
  const tuning_t& tn = tuning();
  int64_t P = 0;
  const double bytes = 4.0 * (double)n_cols * r;
  if (bytes >= 512e6 && n_rows >= 64) {
    // with swept pieces for the panels in between, half as many coarse panels do as well for the
    // gathers and halve the sum over the panels (10,000 x 65.9M, r = 128: 19.8 -> 19.4 ms for both)
    P = (int64_t)ceil(bytes / (sweeps ? 96e6 : 48e6));
    if (P < 8) P = 8;
    if (P > (sweeps ? 256 : 512)) P = sweeps ? 256 : 512;
    const int64_t by_partials = (int64_t)(PANEL_PARTIALS_BYTES / (4.0 * (double)n_rows * r));
    if (P > by_partials) P = by_partials < 8 ? 8 : by_partials;
  }
  if (tn.panels >= 0.0) P = (int64_t)tn.panels;
  if (P > 512) P = 512;
  const int64_t row_groups = ceil_div(n_rows, 4);
  while (P > 1 && P * row_groups >= ((int64_t)1 << 24)) P /= 2;
  return P < 2 ? 0 : P;
}
bool sweeps_for_rank(int r) { return spmm_n_sweep_supported(r) && tuning().sweep_bytes > 0.0 && xcd_round_robin(); }
int max_panels() { return MAX_PANELS; }

static panel_plan panel_policy(const dnpeff_csr* S, int r) {
  const tuning_t& tn = tuning();
  const bool sweeps = sweeps_for_rank(r);
  int64_t P = coarse_panels_for(S->n_rows, S->n_cols, r, sweeps);
  if (S->nnz == 0) P = 0;
  panel_plan plan;
  plan.coarse = (int)P;
  if (P > 0 && sweeps) {
    double sweep_bytes = tn.sweep_bytes;
    if (sweep_bytes > 1e9) sweep_bytes = 1e9;  // (the kernel addresses a piece with 32 bits)
    plan.sweep_cols = (int)(sweep_bytes / (4.0 * sweep_width(r)));  // (a piece of one slice)
    // a piece must also bring work enough for a sweep step (a wait for the other workgroups of
    // the XCD and two barriers): 20,000 entries over all rows
    plan.sweep_min = 4.0;
    if (S->n_rows > 0 && 20000.0 / (double)S->n_rows > plan.sweep_min)
      plan.sweep_min = 20000.0 / (double)S->n_rows;
    if (tn.sweep_min >= 0.0) plan.sweep_min = tn.sweep_min;
    if (plan.sweep_cols <= 0) plan.sweep_cols = 0, plan.sweep_min = 0.0;
  }
  return plan;
}

// The products of a sparse part run on component slices (lists.hip) only when the switches
// n_lists / t_lists ask for it (1): at the sizes measured they are slower than the panels, swept
// pieces and 4-slice column kernel that the plan uses otherwise.  Needs a rank that is a multiple
// of 32 and workgroups dealt to the XCDs round-robin.
bool use_nlists(const dnpeff_csr* S, int r) {
  return tuning().n_lists == 1.0 && nlists_supported(S, r) && xcd_round_robin();
}
// The far tail only (the plain panels past the last swept one) on slot lists, beside the panels
// and swept pieces of the columns before it: n_lists = 2 wherever the lists can be built; left to
// itself (n_lists < 0) where it was measured to pay: ranks from 256 (eight slices or more: one per
// XCD, the entry streams read once per slice) and four rows or more per lane group (with fewer,
// the groups' lists of a piece are short and uneven, and most of a batch is filler): 195 against
// 221 ms for A H^T at 20,000 x 211M, r = 256, 397 against 462 ms at 40,000 ragged rows, r = 512,
// but 20.6 against 19.6 ms at 10,000 rows, r = 128.
bool use_nlists_tail(const dnpeff_csr* S, int r) {
  const double sw = tuning().n_lists;
  if (!(sw == 2.0 || sw < 0.0) || !nlists_supported(S, r) || !xcd_round_robin()) return false;
  if (sw == 2.0) return true;
  return r >= 256 && S->n_rows >= 4 * 8 * (int64_t)nlists_slots(S->n_rows, r);
}
bool use_tlists(const dnpeff_csr* S, int r) {
  return tuning().t_lists > 0.0 && tlists_supported(S, r) && xcd_round_robin();
}

int csr_ensure_products(dnpeff_csr* A, int r) {
  dnpeff_csr* S = sparse_part(A);
  DN_TRY(dnpeff_csr_build_transpose(S));
  if (use_nlists(S, r)) {
    DN_TRY(csr_set_panels(S, panel_plan()));
    DN_TRY(nlists_build(S, r));
  } else {
    panel_plan plan = panel_policy(S, r);
    plan.tail_lists = plan.coarse > 0 && plan.sweep_cols > 0 && use_nlists_tail(S, r) && !S->tail_declined;
    DN_TRY(csr_set_panels(S, plan));
    if (S->tail_floor > 0) {
      // Left to itself, the plan gives the lists what the panel copy of the same entries would
      // take plus half of the memory that the plan keeps free; beyond that the tail stays panels.
      bool declined = false;
      double bound = -1.0;
      if (!(S->nl.pairs && S->nl.floor_col == S->tail_floor)) {  // (lists that exist are not judged again)
        size_t free_b = 0, total_b = 0;
        DN_HIP(hipMemGetInfo(&free_b, &total_b));
        if (tuning().n_lists < 0.0) bound = (double)total_b / 128.0;
        if (tuning().nl_extra_mb >= 0.0) bound = tuning().nl_extra_mb * 1048576.0;
      }
      DN_TRY(nlists_build(S, r, S->tail_floor, bound, &declined));
      if (declined) {
        S->tail_declined = true;  // (later calls must come to the same plan: the matrix may be consumed by then)
        plan.tail_lists = false;
        DN_TRY(csr_set_panels(S, plan));
      }
    } else {
      nlists_drop(S);
    }
  }
  if (use_tlists(S, r)) DN_TRY(tblocks_build(S));
  if (use_spmm_t_bal(S, r)) DN_TRY(fused_tiles_build(S, r));
  DN_TRY(csr_ensure_partials(S, r));
  return head_ensure_workspace(A, r);
}

int csr_consume_for_products(dnpeff_csr* A) {
  DN_HIP(hipStreamSynchronize(stream()));
  dnpeff_csr* S = sparse_part(A);
  if (A->tail) {  // the products read the dense head and the tail, not the whole matrix
    dfree(A->colind); A->colind = nullptr;
    dfree(A->vals); A->vals = nullptr;
    dfree(A->chunk_base); A->chunk_base = nullptr; A->n_chunks = 0;
    dfree(A->partials); A->partials = nullptr; A->partials_floats = 0;
  }
  if ((S->n_panels > 0 || S->nl.pairs) && S->nnz > 0) {  // A H^T reads the regrouped copy / the slot lists
    DN_TRY(csr_ensure_chunks(S));  // (sizes the partial sums; needs the row offsets only)
    dfree(S->colind); S->colind = nullptr;
    dfree(S->vals); S->vals = nullptr;
  }
  return 0;
}

int csr_tile_lists(dnpeff_csr* A) {
  dnpeff_csr* S = sparse_part(A);
  if (S->fused.tiles && S->fused.tile_cols == 32) DN_TRY(fused_tiles_first(S));
  if (A->h_lists_valid) return 0;
  A->h_head_cols.assign((size_t)A->head.n_d, 0);
  A->h_long_cols.assign((size_t)S->n_long, 0);
  DN_HIP(hipStreamSynchronize(stream()));
  if (A->head.n_d)
    DN_HIP(copy_down(A->h_head_cols.data(), A->head.cols, sizeof(int32_t) * A->head.n_d));
  if (S->n_long)
    DN_HIP(copy_down(A->h_long_cols.data(), S->long_cols, sizeof(int32_t) * S->n_long));
  A->h_lists_valid = true;
  return 0;
}

int csr_ensure_partials(dnpeff_csr* A, int r) {
  DN_TRY(csr_ensure_chunks(A));
  int64_t need = A->n_chunks * (int64_t)r;
  if (A->n_panels > 0 && A->n_rows * panel_slots(A) * (int64_t)r > need)
    need = A->n_rows * panel_slots(A) * (int64_t)r;
  if (A->nl.pairs && A->n_rows * (int64_t)r > need) need = A->n_rows * (int64_t)r;
  if (need <= A->partials_floats && A->partials) return 0;
  dfree(A->partials);
  A->partials = nullptr;
  DN_TRY(dmalloc(&A->partials, need));
  A->partials_floats = need;
  return 0;
}

}  // namespace dn

using namespace dn;

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

DN_API const char* dnpeff_last_error(void) { return g_error; }

DN_API int dnpeff_device_count(int* count) {
  DN_CHECK(count != nullptr, "count is NULL");
  int c = 0;
  hipError_t e = hipGetDeviceCount(&c);
  if (e != hipSuccess) c = 0;
  *count = c;
  return 0;
}

DN_API int dnpeff_device_info(char* name, int name_len, int64_t* total_bytes, int* n_cus_out) {
  hipDeviceProp_t p;
  DN_HIP(hipGetDeviceProperties(&p, 0));
  if (name && name_len > 0) {
    strncpy(name, p.name, (size_t)name_len - 1);
    name[name_len - 1] = 0;
  }
  if (total_bytes) *total_bytes = (int64_t)p.totalGlobalMem;
  if (n_cus_out) *n_cus_out = p.multiProcessorCount;
  return 0;
}

DN_API int dnpeff_sync(void) {
  DN_HIP(hipStreamSynchronize(stream()));
  return 0;
}

DN_API void* dnpeff_stream(void) { return (void*)stream(); }

DN_API int dnpeff_tuning_set(const char* name, double value) {
  clear_error();
  DN_CHECK(name != nullptr, "name is NULL");
  for (const tuning_entry& e : g_tuning_table)
    if (strcmp(e.name, name) == 0) {
      tuning().*(e.field) = value;
      return 0;
    }
  DN_CHECK(false, "no tuning switch named '%s'", name);
  return 0;
}

DN_API int dnpeff_tuning_get(const char* name, double* value) {
  clear_error();
  DN_CHECK(name && value, "NULL argument");
  for (const tuning_entry& e : g_tuning_table)
    if (strcmp(e.name, name) == 0) {
      *value = tuning().*(e.field);
      return 0;
    }
  DN_CHECK(false, "no tuning switch named '%s'", name);
  return 0;
}

DN_API int dnpeff_tuning_reset(void) {
  tuning() = tuning_from_env();
  return 0;
}

DN_API int dnpeff_device_memory(int64_t* free_bytes, int64_t* total_bytes) {
  clear_error();
  size_t f = 0, t = 0;
  DN_HIP(hipStreamSynchronize(stream()));
  pool_trim();
  DN_HIP(hipMemGetInfo(&f, &t));
  if (free_bytes) *free_bytes = (int64_t)f;
  if (total_bytes) *total_bytes = (int64_t)t;
  return 0;
}

DN_API int dnpeff_dev_malloc(int64_t bytes, void** out) {
  clear_error();
  DN_CHECK(out != nullptr && bytes >= 0, "bad arguments");
  void* p = nullptr;
  bool reused = false;
  DN_TRY(device_alloc(&p, (size_t)bytes, &reused));
  // (the caller may use the block on any stream: what the library has queued on it must be done)
  if (reused) DN_HIP(hipStreamSynchronize(stream()));
  *out = p;
  return 0;
}

DN_API int dnpeff_dev_free(void* p) {
  if (!p) return 0;
  DN_HIP(hipDeviceSynchronize());  // (work of any stream may still use the block, as for hipFree)
  device_release(p);
  return 0;
}

DN_API int dnpeff_dev_upload(void* dst_dev, const void* src_host, int64_t bytes) {
  clear_error();
  DN_CHECK(bytes >= 0 && (bytes == 0 || (dst_dev && src_host)), "bad arguments");
  DN_HIP(hipStreamSynchronize(stream()));
  DN_HIP(hipStreamSynchronize(nullptr));  // (and for what other blocking streams still do, as hipMemcpy does)
  if (bytes) DN_HIP(copy_up(dst_dev, src_host, (size_t)bytes));
  return 0;
}

DN_API int dnpeff_dev_download(void* dst_host, const void* src_dev, int64_t bytes) {
  clear_error();
  DN_CHECK(bytes >= 0 && (bytes == 0 || (dst_host && src_dev)), "bad arguments");
  DN_HIP(hipStreamSynchronize(stream()));
  DN_HIP(hipStreamSynchronize(nullptr));
  if (bytes) DN_HIP(copy_down(dst_host, src_dev, (size_t)bytes));
  return 0;
}

DN_API int dnpeff_scratch_malloc(int64_t bytes, void** out) {
  clear_error();
  DN_CHECK(out != nullptr && bytes >= 0, "bad arguments");
  return device_alloc(out, (size_t)bytes);
}

DN_API int dnpeff_scratch_free(void* p) {
  device_release(p);
  return 0;
}

DN_API int dnpeff_scratch_download(int n, void* const* dst_host, const void* const* src_dev, const int64_t* bytes) {
  clear_error();
  DN_CHECK(n >= 0 && (n == 0 || (dst_host && src_dev && bytes)), "bad arguments");
  std::vector<copy_part> parts;
  for (int q = 0; q < n; q++) {
    DN_CHECK(bytes[q] >= 0 && (bytes[q] == 0 || (dst_host[q] && src_dev[q])), "bad arguments");
    if (bytes[q]) parts.push_back({dst_host[q], src_dev[q], (size_t)bytes[q]});
  }
  DN_HIP(copy_down_parts(parts.data(), (int)parts.size()));
  return 0;
}

DN_API int64_t dnpeff_size_of_split(int64_t total, int64_t n_splits, int64_t split_index) {
  if (n_splits <= 0 || split_index < 0 || split_index >= n_splits) return -1;
  int64_t base = total / n_splits;
  return split_index == n_splits - 1 ? base + total % n_splits : base;
}

static int validate_host_csr(int64_t n_rows, int64_t n_cols, int64_t nnz, const int64_t* rowptr) {
  DN_CHECK(n_rows >= 0 && n_cols >= 0 && nnz >= 0, "negative matrix dimension");
  DN_CHECK(n_rows < (int64_t)INT32_MAX && n_cols < (int64_t)INT32_MAX,
           "n_rows and n_cols must fit 32-bit ids");
  DN_CHECK(rowptr != nullptr, "rowptr is NULL");
  DN_CHECK(rowptr[0] == 0 && rowptr[n_rows] == nnz, "rowptr[0] must be 0 and rowptr[n_rows] == nnz");
  for (int64_t i = 0; i < n_rows; i++)
    DN_CHECK(rowptr[i] <= rowptr[i + 1], "rowptr decreases at row %lld", (long long)i);
  return 0;
}

__global__ void __launch_bounds__(256)
    k_check_cols(const int32_t* __restrict__ colind, int64_t nnz, int64_t n_cols, int* bad) {
  int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nnz; e += stride) {
    int32_t c = colind[e];
    if (c < 0 || c >= n_cols) atomicAdd(bad, 1);
  }
}

static int check_cols_in_range(const dnpeff_csr* A) {
  int* bad = nullptr;
  DN_TRY(dmalloc(&bad, 1));
  DN_HIP(hipMemsetAsync(bad, 0, sizeof(int), stream()));
  hipLaunchKernelGGL(k_check_cols, dim3(grid_for(A->nnz)), dim3(256), 0, stream(), A->colind,
                     A->nnz, A->n_cols, bad);
  DN_LAUNCH_CHECK();
  int h = 0;
  DN_HIP(copy_down(&h, bad, sizeof(int)));
  dfree(bad);
  DN_CHECK(h == 0, "%d column ids outside [0, n_cols)", h);
  return 0;
}

DN_API int dnpeff_csr_from_host(int64_t n_rows, int64_t n_cols, int64_t nnz, const int64_t* rowptr,
                                const int32_t* colind, const float* vals, dnpeff_csr** out) {
  clear_error();
  DN_CHECK(out != nullptr, "out is NULL");
  *out = nullptr;
  DN_TRY(validate_host_csr(n_rows, n_cols, nnz, rowptr));
  DN_CHECK(nnz == 0 || (colind && vals), "colind/vals are NULL");
  dnpeff_csr* A = new dnpeff_csr();
  A->n_rows = n_rows; A->n_cols = n_cols; A->nnz = nnz; A->full_dense_size = n_cols;
  int s = dmalloc(&A->rowptr, n_rows + 1) || dmalloc(&A->colind, nnz) || dmalloc(&A->vals, nnz);
  if (s) { dnpeff_csr_destroy(A); return 1; }
  hipError_t e = copy_up_parts({{A->rowptr, rowptr, sizeof(int64_t) * (n_rows + 1)},
                                {A->colind, colind, sizeof(int32_t) * nnz},
                                {A->vals, vals, sizeof(float) * nnz}});
  if (e != hipSuccess) {
    set_error("upload of the CSR arrays failed: %s", hipGetErrorString(e));
    dnpeff_csr_destroy(A);
    return 1;
  }
  if (check_cols_in_range(A)) { dnpeff_csr_destroy(A); return 2; }
  *out = A;
  return 0;
}

DN_API int dnpeff_csr_from_pef(int64_t n_rows, int64_t k, int64_t dense_fisher_size,
                               const int32_t* indices, const float* values, dnpeff_csr** out) {
  clear_error();
  DN_CHECK(out != nullptr, "out is NULL");
  *out = nullptr;
  DN_CHECK(n_rows >= 0 && k >= 0 && dense_fisher_size >= 0, "negative dimension");
  DN_CHECK(n_rows < (int64_t)INT32_MAX && dense_fisher_size < (int64_t)INT32_MAX,
           "n_rows and dense_fisher_size must fit 32-bit ids");
  int64_t nnz = n_rows * k;
  DN_CHECK(nnz == 0 || (indices && values), "indices/values are NULL");
  dnpeff_csr* A = new dnpeff_csr();
  A->n_rows = n_rows; A->n_cols = dense_fisher_size; A->nnz = nnz;
  A->full_dense_size = dense_fisher_size;
  int s = dmalloc(&A->rowptr, n_rows + 1) || dmalloc(&A->colind, nnz) || dmalloc(&A->vals, nnz);
  if (s) { dnpeff_csr_destroy(A); return 1; }
  hipLaunchKernelGGL(k_pef_rowptr, dim3(grid_for(n_rows + 1)), dim3(256), 0, stream(), n_rows, k,
                     A->rowptr);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && nnz)
    e = copy_up_parts({{A->colind, indices, sizeof(int32_t) * nnz}, {A->vals, values, sizeof(float) * nnz}});
  if (e != hipSuccess) {
    set_error("upload of the PEF arrays failed: %s", hipGetErrorString(e));
    dnpeff_csr_destroy(A);
    return 1;
  }
  if (check_cols_in_range(A)) { dnpeff_csr_destroy(A); return 2; }
  *out = A;
  return 0;
}

DN_API int dnpeff_csr_normalize_rows(dnpeff_csr* A, const float* norms_host, float eps) {
  clear_error();
  DN_CHECK(A && has_row_major(A), "matrix is NULL or its row-major arrays were released");
  DN_CHECK(norms_host != nullptr || A->n_rows == 0, "norms is NULL");
  if (A->n_rows == 0) return 0;
  float* norms = nullptr;
  DN_TRY(dmalloc(&norms, A->n_rows));
  DN_HIP(copy_up(norms, norms_host, sizeof(float) * A->n_rows));
  unsigned grid = (unsigned)(A->n_rows < 65536 ? A->n_rows : 65536);
  hipLaunchKernelGGL(k_normalize_rows, dim3(grid), dim3(256), 0, stream(), A->rowptr, A->vals,
                     norms, eps, A->n_rows);
  DN_LAUNCH_CHECK();
  dfree(norms);
  drop_derived(A);
  A->sq_norm_valid = false;
  return 0;
}

DN_API int dnpeff_csr_compact_columns(dnpeff_csr* A, int min_count) {
  clear_error();
  DN_CHECK(A && has_row_major(A), "matrix is NULL or its row-major arrays were released");
  drop_derived(A);
  A->sq_norm_valid = false;
  dbuf<uint32_t> mask;
  DN_TRY(mask.alloc(ceil_div(A->n_cols, 32)));
  DN_TRY(column_mask_of_counts(A->colind, A->nnz, A->n_cols, min_count, mask));
  A->full_dense_size = A->n_cols;
  int32_t* new_to_og = nullptr;
  DN_TRY(keep_columns(A, mask, &new_to_og));
  dfree(A->kept);
  A->kept = new_to_og;
  return 0;
}

DN_API int dnpeff_csr_retain_columns(dnpeff_csr* A, const int32_t* kept, int64_t n_kept) {
  clear_error();
  DN_CHECK(A && has_row_major(A), "matrix is NULL or its row-major arrays were released");
  DN_CHECK(n_kept >= 0 && (kept || n_kept == 0), "kept is NULL");
  // (without branches: they took longer than the list's way to the device)
  const int32_t n_cols = (int32_t)A->n_cols;
  int outside = 0, descents = 0;
  if (n_kept) outside = (int)(kept[0] < 0) | (int)(kept[0] >= n_cols);
  for (int64_t i = 1; i < n_kept; i++) {
    outside |= (int)(kept[i] < 0) | (int)(kept[i] >= n_cols);
    descents |= (int)(kept[i] <= kept[i - 1]);
  }
  for (int64_t i = 0; outside && i < n_kept; i++)
    DN_CHECK(kept[i] >= 0 && kept[i] < A->n_cols, "kept[%lld] = %d outside [0, %lld)",
             (long long)i, kept[i], (long long)A->n_cols);
  hipStream_t st = stream();
  drop_derived(A);
  A->sq_norm_valid = false;
  dbuf<int32_t> kept_dev;
  DN_TRY(kept_dev.alloc(n_kept));
  if (n_kept) DN_HIP(copy_up(kept_dev, kept, sizeof(int32_t) * n_kept));
  if (!descents) {  // (a new number is the rank among the kept columns)
    dbuf<uint32_t> mask;
    DN_TRY(mask.alloc(ceil_div(A->n_cols, 32)));
    DN_TRY(column_mask_of_list(kept_dev, n_kept, A->n_cols, mask));
    A->full_dense_size = A->n_cols;
    DN_TRY(keep_columns(A, mask, nullptr));
    dfree(A->kept);
    A->kept = kept_dev.release();
    return 0;
  }
  int32_t* table = nullptr;
  DN_TRY(dmalloc(&table, A->n_cols));
  hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(A->n_cols)), dim3(256), 0, st, table, A->n_cols, -1);
  hipLaunchKernelGGL(k_retain_table, dim3(grid_for(n_kept)), dim3(256), 0, st, kept_dev.p, n_kept,
                     table);
  DN_LAUNCH_CHECK();
  A->full_dense_size = A->n_cols;
  int s = apply_column_table(A, table, n_kept);
  dfree(table);
  if (s) return s;
  dfree(A->kept);
  A->kept = kept_dev.release();
  return 0;
}

DN_API int dnpeff_csr_shape(const dnpeff_csr* A, int64_t* n_rows, int64_t* n_cols, int64_t* nnz) {
  DN_CHECK(A != nullptr, "matrix is NULL");
  if (n_rows) *n_rows = A->n_rows;
  if (n_cols) *n_cols = A->n_cols;
  if (nnz) *nnz = A->nnz;
  return 0;
}

DN_API int dnpeff_csr_full_dense_size(const dnpeff_csr* A, int64_t* out) {
  DN_CHECK(A && out, "NULL argument");
  *out = A->full_dense_size;
  return 0;
}

DN_API int dnpeff_csr_download(const dnpeff_csr* A, int64_t* rowptr, int32_t* colind, float* vals) {
  clear_error();
  DN_CHECK(A && has_row_major(A), "matrix is NULL or its row-major arrays were released");
  DN_HIP(copy_down_parts({{rowptr, A->rowptr, rowptr ? sizeof(int64_t) * (A->n_rows + 1) : 0},
                          {colind, A->colind, colind ? sizeof(int32_t) * A->nnz : 0},
                          {vals, A->vals, vals ? sizeof(float) * A->nnz : 0}}));
  return 0;
}

DN_API int dnpeff_csr_kept_indices(const dnpeff_csr* A, int32_t* new_to_og) {
  clear_error();
  DN_CHECK(A && new_to_og, "NULL argument");
  if (A->kept) {
    if (A->n_cols)
      DN_HIP(copy_down(new_to_og, A->kept, sizeof(int32_t) * A->n_cols));
  } else {
    for (int64_t i = 0; i < A->n_cols; i++) new_to_og[i] = (int32_t)i;
  }
  return 0;
}

DN_API int dnpeff_csr_sq_norm(const dnpeff_csr* A, double* out) {
  clear_error();
  DN_CHECK(A && out, "NULL argument");
  if (A->sq_norm_valid) {
    *out = A->sq_norm;
    return 0;
  }
  // (with a dense head the whole matrix's values only exist in the row-major copy)
  const float* v = A->vals ? A->vals : (A->tail ? nullptr : A->tvals);
  DN_CHECK(v != nullptr || A->nnz == 0, "the row-major copy of the matrix was released before its norm was taken");
  double s = 0.0;
  DN_TRY(dnpeff_op_dot(A->nnz, v, v, &s));
  *out = s;
  dnpeff_csr* M = const_cast<dnpeff_csr*>(A);
  M->sq_norm = s;
  M->sq_norm_valid = true;
  return 0;
}

// rowptr_out[i] = newpos[rowptr[i]]
__global__ void __launch_bounds__(256)
    k_map_rowptr(const int64_t* __restrict__ rowptr, int64_t n_rows, const int64_t* __restrict__ newpos,
                 int64_t* __restrict__ rowptr_out) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i <= n_rows; i += stride)
    rowptr_out[i] = newpos[rowptr[i]];
}

namespace dn {

// Which columns form the dense head.  Candidates are the thresholds thr0, 2 thr0, 4 thr0, ...
// (thr0 = ceil(min_fill n_rows)) and "no head"; a candidate is admissible when its dense blocks
// (n_blocks of them: one where the products read it in both directions, two otherwise) stay
// below a sixth of the device memory; its footprint is the blocks plus both sparse copies of
// the remaining entries (16 bytes each).  The choice is the first admissible candidate
// whose footprint is within `budget` bytes (NO_BUDGET: the first admissible one), else the
// admissible candidate with the smallest footprint (fits = false).
int choose_dense_head(dnpeff_csr* A, double min_fill, double budget, int n_blocks, int rank, int64_t t_run, head_choice* out) {
  *out = head_choice();
  out->footprint = 16.0 * (double)A->nnz;
  out->fits = out->footprint <= budget;
  const int64_t m = A->n_cols, n = A->n_rows;
  if (min_fill <= 0.0 || m == 0 || n == 0 || A->nnz == 0) return 0;
  DN_CHECK(has_row_major(A), "matrix is NULL or its row-major arrays were released");
  hipStream_t st = stream();
  dbuf<int> count;
  dbuf<int32_t> pos;
  dbuf<unsigned long long> zsum;
  DN_TRY(count.alloc(m));
  DN_TRY(pos.alloc(m + 1));
  DN_TRY(zsum.alloc(1));
  DN_TRY(count_columns(A->colind, A->nnz, m, count));
  size_t free_b = 0, total_b = 0;
  DN_HIP(hipMemGetInfo(&free_b, &total_b));
  const int64_t n_pad = ceil_div(n, 128) * 128;
  int64_t thr = (int64_t)ceil(min_fill * (double)n);
  if (thr < 1) thr = 1;
  head_choice best = *out;  // "no head"
  bool have_fit = false;
  // candidates a fifth apart (a doubled threshold can leave a quarter of the budget unused)
  for (; thr <= n && thr <= (int64_t)INT32_MAX; thr = std::max(thr + 1, thr + thr / 5)) {
    int32_t n_d = 0;
    unsigned long long z_head = 0;
    DN_TRY(scan_keep_mask(count, (int)thr, m, pos));
    DN_HIP(copy_down(&n_d, pos + m, sizeof(int32_t)));
    if (n_d == 0) break;
    DN_HIP(hipMemsetAsync(zsum, 0, sizeof(unsigned long long), st));
    hipLaunchKernelGGL(k_sum_selected, dim3(grid_for(m, 4096)), dim3(256), 0, st, count.p, m, (int)thr,
                       zsum.p);
    DN_LAUNCH_CHECK();
    DN_HIP(copy_down(&z_head, zsum, sizeof(unsigned long long)));
    const double blocks = n_blocks * 4.0 * (double)n_pad * (double)(ceil_div(n_d, 128) * 128);
    if (blocks > (double)total_b / 6.0) continue;
    head_choice c;
    c.thr = thr;
    c.n_d = n_d;
    c.z_head = (int64_t)z_head;
    c.footprint = blocks + 16.0 * (double)(A->nnz - (int64_t)z_head) +
                  (rank > 0 ? 4.0 * (double)head_workspace_floats(n, n_d, rank, t_run) : 0.0);
    c.fits = c.footprint <= budget;
    if (c.fits) {
      best = c;
      have_fit = true;
      break;
    }
    if (c.footprint < best.footprint) best = c;
  }
  if (!have_fit && out->fits) return 0;  // no head fits the budget, a head does not
  *out = best;
  return 0;
}

// Moves the columns with at least thr entries into the dense head.
int split_dense_head_at(dnpeff_csr* A, int64_t thr, int64_t* n_dense) {
  hipStream_t st = stream();
  drop_derived(A);
  if (n_dense) *n_dense = 0;
  const int64_t m = A->n_cols, n = A->n_rows;
  if (thr <= 0 || thr > n || m == 0 || A->nnz == 0) return 0;
  DN_CHECK(has_row_major(A), "matrix is NULL or its row-major arrays were released");
  dbuf<int> count;
  dbuf<int32_t> pos, slot_of, cols, table;
  DN_TRY(count.alloc(m));
  DN_TRY(count_columns(A->colind, A->nnz, m, count));
  DN_TRY(pos.alloc(m + 1));
  DN_TRY(scan_keep_mask(count, (int)thr, m, pos));
  int32_t n_d = 0;
  DN_HIP(copy_down(&n_d, pos + m, sizeof(int32_t)));
  if (n_d == 0) return 0;
  const int64_t n_pad = ceil_div(n, 128) * 128, n_d_pad = ceil_div(n_d, 128) * 128;
  DN_TRY(slot_of.alloc(m));
  DN_TRY(cols.alloc((int64_t)n_d));
  DN_TRY(table.alloc(m));
  hipLaunchKernelGGL(k_build_maps, dim3(grid_for(m)), dim3(256), 0, st, count.p, (int)thr, pos.p, m,
                     slot_of.p, cols.p);
  hipLaunchKernelGGL(k_tail_table, dim3(grid_for(m)), dim3(256), 0, st, slot_of.p, m, table.p);
  DN_LAUNCH_CHECK();
  DN_HIP(hipStreamSynchronize(st));
  count.reset();
  pos.reset();
  dbuf<float> cm;
  DN_TRY(cm.alloc(n_d_pad * n_pad));
  DN_HIP(hipMemsetAsync(cm, 0, sizeof(float) * (size_t)(n_d_pad * n_pad), st));
  {
    dbuf<int> repeats;
    DN_TRY(repeats.alloc(1));
    DN_HIP(hipMemsetAsync(repeats, 0, sizeof(int), st));
    hipLaunchKernelGGL(k_head_fill, dim3(grid_for(n * 256)), dim3(256), 0, st, A->rowptr, A->colind,
                       A->vals, n, slot_of.p, cm.p, n_pad, repeats.p);
    DN_LAUNCH_CHECK();
    int n_rep = 0;
    DN_HIP(copy_down(&n_rep, repeats.p, sizeof(int)));
    DN_CHECK(n_rep == 0,
             "%d entries of the dense head's columns repeat a (row, column) pair: duplicate entries are "
             "not supported by the products",
             n_rep);
  }
  // the remaining entries: the row-major arrays without the head's columns, written straight
  // into the tail's own arrays (positions from a scan over the entries)
  dnpeff_csr* T = new dnpeff_csr();
  T->n_rows = n; T->n_cols = m; T->full_dense_size = A->full_dense_size;
  int status = 0;
  {
    dbuf<int64_t> newpos;
    status = newpos.alloc(A->nnz + 1) || scan_kept_entries(A->colind, table, A->nnz, newpos);
    if (!status && copy_down(&T->nnz, newpos + A->nnz, sizeof(int64_t)) != hipSuccess) {
      set_error("dense head: reading the size of the sparse part failed");
      status = 1;
    }
    if (!status)
      status = dmalloc(&T->rowptr, n + 1) || dmalloc(&T->colind, T->nnz) || dmalloc(&T->vals, T->nnz);
    if (!status) {
      hipLaunchKernelGGL(k_compact_entries, dim3(grid_for(A->nnz)), dim3(256), 0, st, A->colind,
                         A->vals, A->nnz, table.p, newpos.p, T->colind, T->vals);
      hipLaunchKernelGGL(k_map_rowptr, dim3(grid_for(n + 1)), dim3(256), 0, st, A->rowptr, n, newpos.p,
                         T->rowptr);
      if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) {
        set_error("dense head: building the sparse part failed");
        status = 1;
      }
    }
  }
  if (status) {
    dnpeff_csr_destroy(T);
    return status;
  }
  dense_head& h = A->head;
  h.n_d = n_d; h.n_d_pad = n_d_pad; h.n_pad = n_pad;
  h.cols = cols.release(); h.cm = cm.release();
  A->tail = T;
  if (n_dense) *n_dense = n_d;
  return 0;
}

}  // namespace dn

DN_API int dnpeff_csr_split_dense_head(dnpeff_csr* A, double min_fill, int64_t* n_dense) {
  clear_error();
  DN_CHECK(A && has_row_major(A), "matrix is NULL or its row-major arrays were released");
  DN_CHECK(min_fill <= 1.0, "min_fill %g above 1", min_fill);
  if (n_dense) *n_dense = 0;
  if (min_fill <= 0.0) {
    drop_derived(A);
    return 0;
  }
  head_choice c;
  DN_TRY(choose_dense_head(A, min_fill, NO_BUDGET, 2, 0, HEAD_RUN, &c));
  return split_dense_head_at(A, c.thr, n_dense);
}

namespace dn {
// Whole tiles per workgroup; few enough workgroups for every one to add up the others' counts.
struct threshold_runs {
  int64_t per_wg;
  unsigned wgs;
  explicit threshold_runs(int64_t count) {
    per_wg = ceil_div(ceil_div(count, THR_TILE), THR_MAX_WGS) * THR_TILE;
    wgs = (unsigned)ceil_div(count, per_wg);
  }
};

static int threshold_write(int64_t count, const float* x, float divisor, float threshold, const int* counts,
                           int32_t* idx_out, float* val_out, unsigned long long* total) {
  const threshold_runs runs(count);
  if (((uintptr_t)x % 16) == 0)
    hipLaunchKernelGGL(k_threshold_write<true>, dim3(runs.wgs), dim3(256), 0, stream(), x, divisor, threshold, count,
                       runs.per_wg, counts, idx_out, val_out, total);
  else
    hipLaunchKernelGGL(k_threshold_write<false>, dim3(runs.wgs), dim3(256), 0, stream(), x, divisor, threshold, count,
                       runs.per_wg, counts, idx_out, val_out, total);
  DN_LAUNCH_CHECK();
  return 0;
}

// The least x with x / divisor >= threshold.  A rounded quotient does not fall as x grows (0 < divisor < infinity), so that
// x >= cut and x / divisor >= threshold are one test; NaN passes neither.  +infinity passes every threshold.
static float threshold_cut(float divisor, float threshold) {
  auto of_key = [](uint32_t key) {  // keys in the order of the floats
    const uint32_t bits = key & 0x80000000u ? key ^ 0x80000000u : ~key;
    float f;
    std::memcpy(&f, &bits, 4);
    return f;
  };
  uint32_t lo = 0x007fffffu, hi = 0xff800000u;  // -infinity, +infinity
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (of_key(mid) / divisor >= threshold) hi = mid;
    else lo = mid + 1;
  }
  return of_key(hi);
}

// What dnpeff_threshold_find leaves for dnpeff_threshold_take: in the pinned buffer (positions, then values), or on
// the device.
struct threshold_found {
  pinned_buf pinned;
  dbuf<int32_t> idx;
  dbuf<float> val;
  int64_t n = 0;
  bool at_hand = false;
  hipStream_t st = nullptr;
  ~threshold_found() {  // (nothing may still be on its way to the buffer)
    if (st) (void)hipStreamSynchronize(st);
  }
};
}  // namespace dn

DN_API int dnpeff_op_threshold_compact(int64_t count, const float* x, float divisor, float threshold,
                                       int32_t* idx_out, float* val_out, int64_t* n_kept) {
  clear_error();
  DN_CHECK(count >= 0 && count <= (int64_t)INT32_MAX, "count %lld outside [0, 2^31)", (long long)count);
  DN_CHECK((x && idx_out && val_out) || count == 0, "NULL argument");
  DN_CHECK(n_kept != nullptr, "n_kept is NULL");
  DN_CHECK(divisor != 0.0f, "divisor is zero");
  *n_kept = 0;
  if (count == 0) return 0;
  const threshold_runs runs(count);
  dbuf<int> counts;
  DN_TRY(counts.alloc(runs.wgs));
  unsigned long long* total = nullptr;
  DN_TRY(host_words(&total));
  hipStream_t st = stream();
  if (((uintptr_t)x % 16) == 0)
    hipLaunchKernelGGL(k_threshold_count<true>, dim3(runs.wgs), dim3(256), 0, st, x, divisor, threshold, count,
                       runs.per_wg, counts.p);
  else
    hipLaunchKernelGGL(k_threshold_count<false>, dim3(runs.wgs), dim3(256), 0, st, x, divisor, threshold, count,
                       runs.per_wg, counts.p);
  DN_TRY(threshold_write(count, x, divisor, threshold, counts.p, idx_out, val_out, total));
  DN_HIP(hipStreamSynchronize(st));
  *n_kept = (int64_t)*total;
  return 0;
}

DN_API int dnpeff_threshold_find(int64_t count, const float* x, float divisor, float threshold, int64_t* n_kept,
                                 void** found) {
  clear_error();
  DN_CHECK(count >= 0 && count <= (int64_t)INT32_MAX, "count %lld outside [0, 2^31)", (long long)count);
  DN_CHECK(x || count == 0, "NULL argument");
  DN_CHECK(n_kept != nullptr && found != nullptr, "n_kept or found is NULL");
  DN_CHECK(divisor != 0.0f, "divisor is zero");
  *n_kept = 0;
  *found = nullptr;
  std::unique_ptr<threshold_found> F(new (std::nothrow) threshold_found);
  DN_CHECK(F != nullptr, "out of host memory");
  if (count > 0) {
    const threshold_runs runs(count);
    dbuf<int> counts;
    dbuf<uint2> notes;
    DN_TRY(counts.alloc(runs.wgs));
    DN_TRY(notes.alloc((int64_t)runs.wgs * THR_KEEP));
    unsigned long long* word = nullptr;
    DN_TRY(host_waited_words(&word));
    *word = WORD_NONE;
    F->pinned.take();
    constexpr int ROOM = (int)(pinned_buf::BYTES / 8);
    hipStream_t st = F->st = stream();
    const bool vec4 = ((uintptr_t)x % 16) == 0, by_cut = divisor > 0.0f && divisor < INFINITY && threshold == threshold;
    const auto find = vec4 ? by_cut ? k_threshold_find<true, true> : k_threshold_find<true, false>
                           : by_cut ? k_threshold_find<false, true> : k_threshold_find<false, false>;
    hipLaunchKernelGGL(find, dim3(runs.wgs), dim3(256), 0, st, x, divisor,
                       by_cut ? threshold_cut(divisor, threshold) : threshold, count, runs.per_wg, counts.p, notes.p);
    hipLaunchKernelGGL(k_threshold_pack, dim3(ROOM / 1024), dim3(256), 0, st, counts.p, (int)runs.wgs, notes.p,
                       divisor, F->pinned.p() ? ROOM : 0, (int4*)F->pinned.p(),
                       (float4*)(F->pinned.p() ? F->pinned.p() + 4 * ROOM : nullptr), word);
    DN_LAUNCH_CHECK();
    // (the finds are still on their way: the caller makes room for them meanwhile.  4 components of 6 M: 283 -> 277 us, a first time
    // 331 -> 309)
    DN_HIP(wait_words(word, 1, st));
    F->n = (int64_t)(*word & (THR_FITS - 1));
    F->at_hand = (*word & THR_FITS) != 0;
    if (!F->at_hand) {
      DN_TRY(F->idx.alloc(F->n));
      DN_TRY(F->val.alloc(F->n));
      DN_TRY(threshold_write(count, x, divisor, threshold, counts.p, F->idx.p, F->val.p, nullptr));
      DN_HIP(hipStreamSynchronize(st));  // (x is the caller's again)
    }
  }
  *n_kept = F->n;
  *found = F.release();
  return 0;
}

DN_API int dnpeff_threshold_take(void* found, int32_t* idx_host, float* val_host) {
  clear_error();
  std::unique_ptr<threshold_found> F((threshold_found*)found);
  DN_CHECK(F != nullptr, "found is NULL");
  const size_t bytes = 4 * (size_t)F->n;
  if (!bytes || (!idx_host && !val_host)) return 0;
  DN_CHECK(idx_host && val_host, "NULL argument");
  if (F->at_hand) {
    fetch_pages(idx_host, bytes);
    fetch_pages(val_host, bytes);
    DN_HIP(hipStreamSynchronize(F->st));
    std::memcpy(idx_host, F->pinned.p(), bytes);
    std::memcpy(val_host, F->pinned.p() + pinned_buf::BYTES / 2, bytes);
  } else {
    DN_HIP(copy_down_parts({{idx_host, F->idx.p, bytes}, {val_host, F->val.p, bytes}}));
  }
  return 0;
}

DN_API int dnpeff_csr_head_info(const dnpeff_csr* A, int64_t* n_dense, int64_t* nnz_sparse) {
  DN_CHECK(A != nullptr, "matrix is NULL");
  if (n_dense) *n_dense = A->head.n_d;
  if (nnz_sparse) *nnz_sparse = sparse_part(A)->nnz;
  return 0;
}

DN_API int dnpeff_csr_products_info(const dnpeff_csr* A, int64_t* out6) {
  DN_CHECK(A != nullptr && out6 != nullptr, "NULL argument");
  const dnpeff_csr* S = sparse_part(A);
  out6[0] = S->n_panels;
  out6[1] = S->n_plain;
  out6[2] = S->n_swept;
  out6[3] = S->tail_floor;
  out6[4] = S->nl.pairs ? S->nl.n_entries : 0;
  out6[5] = S->nl.pairs ? S->nl.n_batches : 0;
  return 0;
}

// A launch per row takes 3.5 us and the check for repeated rows reads every column again.  With bits an
// entry reads the words of its column below its own, up to 64 of them, which pays while the bits stay in the
// memory-side cache (300 rows, 0.6 M entries, 145 k columns: 1280 -> 152 us; 2000 rows, 4 M entries, 100 k columns:
// 7.6 -> 0.93 ms; with 435 MB of bits, 1000 rows, 16.4 M entries: 6.0 and 6.4 ms).
static bool transpose_bits_pay(const dnpeff_csr* A) {
  return A->n_rows <= 2048 && A->nnz > 0 &&
         4 * ceil_div(A->n_rows, 32) * A->n_cols <= ((int64_t)128 << 20);
}

// *done = false: a row holds a column twice.
static int transpose_by_bits(const dnpeff_csr* A, int* count, int64_t* colptr, int32_t* rowind, float* tvals, bool* done) {
  hipStream_t st = stream();
  const int64_t m = A->n_cols, n = A->n_rows;
  const int words = (int)ceil_div(n, 32);
  dbuf<uint32_t> bits;
  DN_TRY(bits.alloc(m * words));
  unsigned long long* host = nullptr;
  DN_TRY(host_words(&host));
  int64_t* total = reinterpret_cast<int64_t*>(host);
  DN_HIP(hipMemsetAsync(bits, 0, sizeof(uint32_t) * (size_t)(m * words), st));
  const int64_t per_row = std::min<int64_t>(64, std::max<int64_t>(1, ceil_div(ceil_div(A->nnz, n), 1024)));
  const dim3 grid((unsigned)per_row, (unsigned)n), block(256);
  hipLaunchKernelGGL(k_bits_set, grid, block, 0, st, A->rowptr, A->colind, n, words, bits.p);
  hipLaunchKernelGGL(k_bits_count, dim3(grid_for(m)), block, 0, st, bits.p, words, m, count);
  DN_LAUNCH_CHECK();
  DN_TRY(scan_counts_i64(count, m, colptr, total));
  DN_HIP(hipStreamSynchronize(st));
  *done = *total == A->nnz;  // (an entry that repeats sets no bit of its own)
  if (!*done) return 0;
  hipLaunchKernelGGL(k_bits_place, grid, block, 0, st, A->rowptr, A->colind, A->vals, n, bits.p, words, colptr, rowind,
                     tvals);
  DN_LAUNCH_CHECK();
  return 0;
}

// Where a row has an entry per range or more on average: the table has four bytes for each.  (Most lanes have no entry then:
// 0.6 ms at 2.8 M entries of 256 rows and 22 M columns as at 11 M, but 1.8 and 2.8 row by row.)  Whole builds of the
// transposed copy, row by row / by ranges: 256 rows, 22 M columns, 56 M entries 9.4 / 1.05 ms, 22 M 4.5 / 0.7, 1000 rows, 4 M
// columns, 20 M entries 5.6 / 1.2, 4 M 3.6 / 0.4, 2100 rows, 0.3 M columns, 6 M entries 7.0 / 0.6.
static bool transpose_ranges_pay(const dnpeff_csr* A) {
  return A->nnz >= ((int64_t)1 << 20) && A->n_rows < ((int64_t)1 << 16) && A->n_cols >= ((int64_t)1 << 18) &&
         (double)A->nnz / (double)A->n_rows * RANGE_COLS >= (double)A->n_cols;
}

// *done = false: the columns of a row do not ascend, or a range has more entries than its counters hold.
static int transpose_by_ranges(const dnpeff_csr* A, int64_t* colptr, int32_t* rowind, float* tvals, bool* done) {
  hipStream_t st = stream();
  const int64_t n = A->n_rows, m = A->n_cols, ranges = ceil_div(m, RANGE_COLS);
  unsigned long long* host = nullptr;
  DN_TRY(host_words(&host));
  int* unfit = reinterpret_cast<int*>(host);
  *unfit = 0;
  hipLaunchKernelGGL(k_range_probe, dim3((unsigned)n), dim3(256), 0, st, A->rowptr, A->colind, unfit);
  DN_LAUNCH_CHECK();
  DN_HIP(hipStreamSynchronize(st));
  if (*unfit) return 0;
  dbuf<uint32_t> at;
  dbuf<int> count;
  dbuf<int64_t> base;
  if (at.alloc((ranges + 1) * n) || count.alloc(ranges + 1) || base.alloc(ranges + 1)) {  // (no room: row by row)
    clear_error();
    return 0;
  }
  const int64_t per_row = std::max<int64_t>(1, std::min<int64_t>(64, A->nnz / n / 1024));
  DN_HIP(hipMemsetAsync(count, 0, sizeof(int), st));  // (its first element: whether columns are out of order)
  hipLaunchKernelGGL(k_range_starts, dim3((unsigned)n, (unsigned)per_row), dim3(256), 0, st, A->rowptr, A->colind, n, ranges,
                     at.p, count.p);
  hipLaunchKernelGGL(k_range_counts, dim3((unsigned)ranges), dim3(256), 0, st, at.p, n, count.p + 1, count.p, unfit);
  DN_LAUNCH_CHECK();
  DN_TRY(scan_counts_i64(count.p + 1, ranges, base));
  DN_HIP(hipStreamSynchronize(st));
  *done = *unfit == 0;
  if (!*done) return 0;
  DN_HIP(hipFuncSetAttribute((const void*)k_range_transpose, hipFuncAttributeMaxDynamicSharedMemorySize, (int)RANGE_LDS));
  hipLaunchKernelGGL(k_range_transpose, dim3((unsigned)ranges), dim3(64 * RANGE_WAVES), RANGE_LDS, st, A->rowptr, A->colind,
                     A->vals, n, m, at.p, base.p, colptr, rowind, tvals);
  DN_LAUNCH_CHECK();
  return 0;
}

// Row by row: the entries of a row have no order among each other.
static int transpose_by_rows(const dnpeff_csr* A, int* count, int64_t* colptr, int32_t* rowind, float* tvals) {
  hipStream_t st = stream();
  const int64_t m = A->n_cols;
  DN_TRY(count_columns(A->colind, A->nnz, m, count));
  DN_TRY(scan_counts_i64(count, m, colptr));
  // (the last element counts columns with a repeated row)
  DN_HIP(hipMemsetAsync(count, 0, sizeof(int) * (size_t)(m + 1), st));
  std::vector<int64_t> rowptr((size_t)A->n_rows + 1);
  DN_HIP(copy_down(rowptr.data(), A->rowptr, sizeof(int64_t) * (A->n_rows + 1)));
  for (int64_t i = 0; i < A->n_rows; i++) {
    int64_t len = rowptr[i + 1] - rowptr[i];
    if (len <= 0) continue;
    hipLaunchKernelGGL(k_transpose_row, dim3((unsigned)ceil_div(len, 256)), dim3(256), 0, st,
                       (int32_t)i, rowptr[i], rowptr[i + 1], A->colind, A->vals, colptr, count, rowind, tvals);
  }
  DN_LAUNCH_CHECK();
  // A row that holds a column twice puts two entries of that row next to each other in the
  // column's list, in an order that the hardware decides: such a matrix has no deterministic
  // transposed copy (nor is it a valid PEF matrix: top-k indices are distinct) and is refused.
  hipLaunchKernelGGL(k_check_repeats, dim3(grid_for(m, 65536)), dim3(256), 0, st, colptr, rowind, m, count + m);
  DN_LAUNCH_CHECK();
  int repeats = 0;
  DN_HIP(copy_down(&repeats, count + m, sizeof(int)));
  DN_CHECK(repeats == 0,
           "%d column(s) hold the same row more than once: duplicate (row, column) entries are not "
           "supported by the products",
           repeats);
  return 0;
}

DN_API int dnpeff_csr_build_transpose(dnpeff_csr* A) {
  clear_error();
  DN_CHECK(A != nullptr, "matrix is NULL");
  if (A->colptr) return 0;
  DN_CHECK(has_row_major(A), "row-major copy of the matrix was released");
  hipStream_t st = stream();
  const int64_t m = A->n_cols;
  dbuf<int> count;
  dbuf<int64_t> colptr;
  dbuf<int32_t> rowind, pos, long_cols;
  dbuf<float> tvals;
  DN_TRY(count.alloc(m + 1));
  DN_TRY(colptr.alloc(m + 1));
  DN_TRY(rowind.alloc(A->nnz));
  DN_TRY(tvals.alloc(A->nnz));
  bool done = false;
  if (transpose_bits_pay(A)) DN_TRY(transpose_by_bits(A, count, colptr, rowind, tvals, &done));
  if (!done && transpose_ranges_pay(A)) DN_TRY(transpose_by_ranges(A, colptr, rowind, tvals, &done));
  if (!done) DN_TRY(transpose_by_rows(A, count, colptr, rowind, tvals));
  count.reset();
  // list of long columns for A^T W; a column has no row twice, so that few rows have none (22 M columns: 0.22 ms)
  int64_t n_long = 0;
  if (A->n_rows > SPMM_T_LONG) {
    DN_TRY(pos.alloc(m + 1));
    unsigned long long* host = nullptr;
    DN_TRY(host_words(&host));
    int64_t* total = reinterpret_cast<int64_t*>(host);
    DN_TRY(scan_long_cols(colptr, SPMM_T_LONG, m, pos, total));
    DN_HIP(hipStreamSynchronize(st));
    n_long = *total;
  } else {
    DN_HIP(hipStreamSynchronize(st));
  }
  DN_TRY(long_cols.alloc(n_long));
  if (n_long) {
    hipLaunchKernelGGL(k_collect_long, dim3(grid_for(m)), dim3(256), 0, st, colptr.p, SPMM_T_LONG, m,
                       pos.p, long_cols.p);
    DN_LAUNCH_CHECK();
  }
  A->colptr = colptr.release();
  A->rowind = rowind.release();
  A->tvals = tvals.release();
  A->long_cols = long_cols.release();
  A->n_long = n_long;
  A->h_lists_valid = false;
  return 0;
}

DN_API int dnpeff_csr_download_transpose(dnpeff_csr* A, int64_t* colptr, int32_t* rowind,
                                         float* vals) {
  clear_error();
  DN_TRY(dnpeff_csr_build_transpose(A));
  if (colptr)
    DN_HIP(copy_down(colptr, A->colptr, sizeof(int64_t) * (A->n_cols + 1)));
  if (rowind && A->nnz)
    DN_HIP(copy_down(rowind, A->rowind, sizeof(int32_t) * A->nnz));
  if (vals && A->nnz)
    DN_HIP(copy_down(vals, A->tvals, sizeof(float) * A->nnz));
  return 0;
}

// out[k] = X[rows[k]] for k < count (rows of r floats)
__global__ void __launch_bounds__(256)
    k_gather_rows(const float* __restrict__ X, const int32_t* __restrict__ rows, int64_t count, int r,
                  float* __restrict__ out) {
  const int64_t total = count * r, stride = (int64_t)gridDim.x * 256;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += stride)
    out[e] = X[(int64_t)rows[e / r] * r + e % r];
}

DN_API int dnpeff_op_gather_rows(int64_t count, int r, const float* X, const int32_t* rows_dev,
                                 float* out) {
  clear_error();
  DN_CHECK(count >= 0 && r >= 1, "bad arguments");
  if (count == 0) return 0;
  DN_CHECK(X && rows_dev && out, "NULL argument");
  hipLaunchKernelGGL(k_gather_rows, dim3(grid_for(count * r)), dim3(256), 0, stream(), X, rows_dev,
                     count, r, out);
  DN_LAUNCH_CHECK();
  return 0;
}

// out[k] = cm[k * n_pad + row]: one row of the dense head's block
__global__ void __launch_bounds__(256)
    k_head_row(const float* __restrict__ cm, int64_t n_pad, int64_t row, int64_t n_d,
               float* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n_d; k += stride)
    out[k] = cm[k * n_pad + row];
}

// Entries of one row / one column of the matrix as the products hold it: the dense head's block
// plus the sparse part (its regrouped or plain row-major copy, its transposed copy).
DN_API int dnpeff_csr_get_row(dnpeff_csr* A, int64_t row, int64_t cap, int64_t* count, int32_t* cols,
                              float* vals) {
  clear_error();
  DN_CHECK(A && count, "NULL argument");
  DN_CHECK(row >= 0 && row < A->n_rows, "row %lld outside [0, %lld)", (long long)row,
           (long long)A->n_rows);
  DN_HIP(hipStreamSynchronize(stream()));
  const dnpeff_csr* S = sparse_part(A);
  DN_CHECK(S->rowptr != nullptr, "matrix has no row offsets");
  int64_t e[2];
  DN_HIP(copy_down(e, S->rowptr + row, sizeof(e)));
  const int32_t* src_c = S->colind ? S->colind : S->pcol;
  const float* src_v = S->vals ? S->vals : S->pval;
  std::vector<int32_t> list_cols;
  std::vector<float> list_vals;
  const int64_t row_entries = e[1] - e[0];
  if (!S->colind && S->pcol && S->tail_floor > 0 && S->nl.pairs) {
    // the panels hold the row's entries below tail_floor, the slot lists the others
    DN_TRY(nlists_get_row(S, row, list_cols, list_vals));
    DN_HIP(copy_down(e, S->prow + row, sizeof(e)));
    DN_CHECK((int64_t)list_cols.size() + (e[1] - e[0]) == row_entries,
             "panels and slot lists hold %lld entries of row %lld, not %lld",
             (long long)((int64_t)list_cols.size() + (e[1] - e[0])), (long long)row, (long long)row_entries);
    std::vector<int32_t> pc((size_t)(e[1] - e[0]));
    std::vector<float> pv((size_t)(e[1] - e[0]));
    if (e[1] > e[0]) {
      DN_HIP(copy_down(pc.data(), S->pcol + e[0], sizeof(int32_t) * pc.size()));
      DN_HIP(copy_down(pv.data(), S->pval + e[0], sizeof(float) * pv.size()));
    }
    list_cols.insert(list_cols.begin(), pc.begin(), pc.end());
    list_vals.insert(list_vals.begin(), pv.begin(), pv.end());
  } else if (!(src_c && src_v) && S->nl.pairs) {  // the sparse part is held as slot lists
    DN_TRY(nlists_get_row(S, row, list_cols, list_vals));
    DN_CHECK((int64_t)list_cols.size() == row_entries, "slot lists hold %lld entries of row %lld, not %lld",
             (long long)list_cols.size(), (long long)row, (long long)row_entries);
  } else {
    DN_CHECK(e[1] == e[0] || (src_c && src_v), "matrix holds no row-major copy of its sparse part");
  }
  int64_t got = row_entries;
  std::vector<float> head_row;
  std::vector<int32_t> head_cols;
  if (A->head.n_d) {
    head_row.resize((size_t)A->head.n_d);
    head_cols.resize((size_t)A->head.n_d);
    dbuf<float> tmp;
    DN_TRY(tmp.alloc(A->head.n_d));
    hipLaunchKernelGGL(k_head_row, dim3(grid_for(A->head.n_d, 4096)), dim3(256), 0, stream(), A->head.cm,
                       A->head.n_pad, row, A->head.n_d, tmp.p);
    DN_LAUNCH_CHECK();
    DN_HIP(hipStreamSynchronize(stream()));
    DN_HIP(copy_down(head_row.data(), tmp.p, sizeof(float) * A->head.n_d));
    DN_HIP(copy_down(head_cols.data(), A->head.cols, sizeof(int32_t) * A->head.n_d));
    for (float v : head_row) got += v != 0.0f;
  }
  *count = got;
  if (!cols || !vals) return 0;
  DN_CHECK(cap >= got, "row %lld holds %lld entries, the buffers %lld", (long long)row, (long long)got,
           (long long)cap);
  int64_t w = 0;
  for (size_t k = 0; k < head_row.size(); k++)
    if (head_row[k] != 0.0f) {
      cols[w] = head_cols[k];
      vals[w++] = head_row[k];
    }
  if (!list_cols.empty()) {
    memcpy(cols + w, list_cols.data(), sizeof(int32_t) * list_cols.size());
    memcpy(vals + w, list_vals.data(), sizeof(float) * list_vals.size());
  } else if (e[1] > e[0]) {
    DN_HIP(copy_down(cols + w, src_c + e[0], sizeof(int32_t) * (e[1] - e[0])));
    DN_HIP(copy_down(vals + w, src_v + e[0], sizeof(float) * (e[1] - e[0])));
  }
  return 0;
}

DN_API int dnpeff_csr_get_column(dnpeff_csr* A, int64_t col, int64_t cap, int64_t* count,
                                 int32_t* rows, float* vals) {
  clear_error();
  DN_CHECK(A && count, "NULL argument");
  DN_CHECK(col >= 0 && col < A->n_cols, "column %lld outside [0, %lld)", (long long)col,
           (long long)A->n_cols);
  dnpeff_csr* S = sparse_part(A);
  DN_TRY(dnpeff_csr_build_transpose(S));
  DN_TRY(csr_tile_lists(A));
  DN_HIP(hipStreamSynchronize(stream()));
  const std::vector<int32_t>& hc = A->h_head_cols;
  const auto it = std::lower_bound(hc.begin(), hc.end(), (int32_t)col);
  if (it != hc.end() && *it == (int32_t)col) {  // a column of the dense head
    const int64_t k = it - hc.begin();
    std::vector<float> c((size_t)A->n_rows);
    DN_HIP(copy_down(c.data(), A->head.cm + k * A->head.n_pad, sizeof(float) * A->n_rows));
    int64_t got = 0;
    for (float v : c) got += v != 0.0f;
    *count = got;
    if (!rows || !vals) return 0;
    DN_CHECK(cap >= got, "column %lld holds %lld entries, the buffers %lld", (long long)col,
             (long long)got, (long long)cap);
    int64_t w = 0;
    for (int64_t i = 0; i < A->n_rows; i++)
      if (c[(size_t)i] != 0.0f) {
        rows[w] = (int32_t)i;
        vals[w++] = c[(size_t)i];
      }
    return 0;
  }
  int64_t p[2];
  DN_HIP(copy_down(p, S->colptr + col, sizeof(p)));
  *count = p[1] - p[0];
  if (!rows || !vals) return 0;
  DN_CHECK(cap >= p[1] - p[0], "column %lld holds %lld entries, the buffers %lld", (long long)col,
           (long long)(p[1] - p[0]), (long long)cap);
  if (p[1] > p[0]) {
    DN_HIP(copy_down(rows, S->rowind + p[0], sizeof(int32_t) * (p[1] - p[0])));
    DN_HIP(copy_down(vals, S->tvals + p[0], sizeof(float) * (p[1] - p[0])));
  }
  return 0;
}

DN_API int dnpeff_csr_release(dnpeff_csr* A, int which) {
  clear_error();
  DN_CHECK(A != nullptr, "matrix is NULL");
  DN_HIP(hipStreamSynchronize(stream()));
  if (which == 1) {
    dfree(A->colind); A->colind = nullptr;
    dfree(A->vals); A->vals = nullptr;
    dfree(A->rowptr); A->rowptr = nullptr;
    dfree(A->chunk_base); A->chunk_base = nullptr; A->n_chunks = 0;
    dfree(A->partials); A->partials = nullptr; A->partials_floats = 0;
  } else if (which == 2) {
    dfree(A->colptr); A->colptr = nullptr;
    dfree(A->rowind); A->rowind = nullptr;
    dfree(A->tvals); A->tvals = nullptr;
    drop_slots(A);
    dfree(A->long_cols); A->long_cols = nullptr; A->n_long = 0;
  } else {
    DN_CHECK(false, "which must be 1 (row-major copy) or 2 (transposed copy)");
  }
  return 0;
}

DN_API int dnpeff_csr_destroy(dnpeff_csr* A) {
  if (!A) return 0;
  (void)hipStreamSynchronize(stream());
  drop_derived(A);
  dfree(A->rowptr);
  dfree(A->colind);
  dfree(A->vals);
  dfree(A->kept);
  delete A;
  return 0;
}
