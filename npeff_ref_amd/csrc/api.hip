// Handles of the two hot loops behind the C ABI: the dense-factor MU NMF of
// run_nmf_on_pefs and the W-only learner of fit_coeffs_to_sparse_H.
#include <chrono>
#include "dnpeff_internal.hpp"
#include "fused.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <utility>
#include <vector>

using namespace dn;

// ---------------------------------------------------------------------------
// Per-kernel timing with HIP events on the library stream
// ---------------------------------------------------------------------------
// A mark is one event on the stream; the time from a mark to the next one belongs to the class
// that the mark opens (none for a mark that only closes).  Classes that follow one another
// without anything between them share the mark between them (next()).
struct Mark {
  hipEvent_t ev = nullptr;
  int cls = -1;
  bool counts = true;  // the segment is a launch of its class (not the continuation of one)
};

struct Profiler {
  bool enabled = false;
  std::vector<Mark> pool;        // every event ever created
  size_t used = 0;               // marks in flight since the last collect
  double ms_sum[DNPEFF_K_COUNT] = {0};
  int64_t launches[DNPEFF_K_COUNT] = {0};

  int mark(int cls, bool counts = true) {
    if (used == pool.size()) {
      Mark m;
      DN_HIP(hipEventCreate(&m.ev));
      pool.push_back(m);
    }
    pool[used].cls = cls;
    pool[used].counts = counts;
    DN_HIP(hipEventRecord(pool[used].ev, stream()));
    used++;
    return 0;
  }
  int begin(int cls) { return enabled ? mark(cls) : 0; }
  // goes on with a class that was interrupted (its time, not another launch)
  int resume(int cls) { return enabled ? mark(cls, false) : 0; }
  // closes the open class and opens cls with the same event
  int next(int cls) { return enabled ? mark(cls) : 0; }
  int end() {
    if (!enabled) return 0;
    DN_TRY(mark(-1));
    if (used >= 32768) return collect();
    return 0;
  }
  int collect() {
    if (used == 0) return 0;
    DN_HIP(hipStreamSynchronize(stream()));
    for (size_t i = 0; i + 1 < used; i++) {
      if (pool[i].cls < 0) continue;
      float ms = 0.0f;
      DN_HIP(hipEventElapsedTime(&ms, pool[i].ev, pool[i + 1].ev));
      if (ms < 0.0f) ms = 0.0f;  // (marks on two streams: the later mark's work ended first)
      ms_sum[pool[i].cls] += (double)ms;
      if (pool[i].counts) launches[pool[i].cls] += 1;
    }
    used = 0;
    return 0;
  }
  void reset() {
    for (int i = 0; i < DNPEFF_K_COUNT; i++) {
      ms_sum[i] = 0.0;
      launches[i] = 0;
    }
  }
  ~Profiler() {
    for (auto& m : pool)
      if (m.ev) (void)hipEventDestroy(m.ev);
  }
};

// ---------------------------------------------------------------------------
// Dense-factor MU NMF
// ---------------------------------------------------------------------------
struct dnpeff_nmf {
  dnpeff_csr* A = nullptr;
  int r = 0;                 // components a row of the factors has in memory
  // The rank.  Ranks above 128 that are not multiples of 128 are stored with zero components up to the
  // next one (padded_rank): the updates keep those zero, and every kernel made for multiples of 128
  // runs.  The factors that callers see are packed.
  int rl = 0;
  float* Wp = nullptr;       // packed copies handed out by dnpeff_nmf_device_factors, while r != rl: they
  float* Hp = nullptr;       // are the factors as long as their pointers are out (take_back, show)
  float eps = 0.0f;
  uint64_t seed = 0;
  int64_t n = 0, m = 0;
  float* W = nullptr;        // [n, r]
  float* W2 = nullptr;       // [n, r] output buffer of the W update
  float* Nw = nullptr;       // [n, r] A H^T
  float* H = nullptr;        // [m, r] (points into Hbuf)
  float* S = nullptr;        // [m, r] A^T W, then the updated H; tiled: [tile_cols, r], A^T W of a tile
  float* S2 = nullptr;       // tiled, h_overlap: a second tile buffer
  float* Hbuf = nullptr;     // allocation that holds H; tiled: [m + tile_cols, r]
  // Tiled H update (when a second [m, r] array does not fit): A^T W is formed for tile_cols
  // columns at a time and the updated tile is written one tile below (or above) the place of the
  // old one inside Hbuf, so the update needs no full-size output: H alternates between
  // Hbuf and Hbuf + tile_cols r.
  bool tiled = false;
  int64_t tile_cols = 0;
  float* G = nullptr;        // [r, r]
  float* G2 = nullptr;       // [r, r]
  float* gram_ws = nullptr;  // slice partials of the Gram kernel
  double* dot_ws = nullptr;  // DOT_BLOCKS partials + 2 results
  float* GH = nullptr;       // [r, r] H^T H from the fused H update (valid while gh_valid)
  float* gpart = nullptr;    // its partial sums
  bool gh_valid = false;
  bool nw_valid = false;     // Nw holds A H^T of the current H (left there by the loss)
  double sq_norm_A = 0.0;
  Profiler prof;
  // The step of small ranks (fused.hip).  While the switch is off, another context's dense head is on
  // the matrix or the launches of each class are being timed, the separate kernels run instead.
  bool has_fused = false;
  fused_state fu;            // (fu.xcd: the memory plan had room for the lists by XCD)
  bool fu_n_valid = false;   // fu.n_part (or Nw, with panels) holds A H^T of the current H
  // The factor's device pointer was handed out since its last update: the caller may write through it
  // between any two calls, so no product kept from an earlier call stands for the factor.
  bool w_out = false, h_out = false;
};

// Rows that one fp32 sum may take in at padded ranks, in X^T X and in the dense head's A^T W.  As they are, those
// ranks sum over a 2048th part of the rows, or 500 of them: left to fill the chip alone, the tiles would sum over
// many times that.  Errors against 64 bits of one update, as they are / padded / padded with these bounds: W at
// 2000 x 3.9 M, r = 385 4.3e-6 / 1.0e-5 / 4.7e-7, H at 2000 x 0.4 M, r = 150 2.5e-7 / 4.5e-7 / 2.2e-7.  Ten
// iterations take 247 against 239 ms there, 28.6 against 28.4, 66.6 against 64.3 at 700 x 1.0 M, r = 500.
constexpr int64_t PADDED_GRAM_RUN = 1024, PADDED_HEAD_RUN = 512;
static int64_t gram_run(const dnpeff_nmf* h) { return h->r != h->rl ? PADDED_GRAM_RUN : 0; }
static int64_t head_run(int rank, int asked) { return rank != asked ? PADDED_HEAD_RUN : HEAD_RUN; }

// At the start of every call that uses the factors: those whose pointers are out are what the caller
// has left there (packed copies are copied back), and what is kept of them is forgotten.
static int take_back(dnpeff_nmf* h) {
  const bool packed = h->r != h->rl;
  if (h->w_out) {
    if (packed) DN_TRY(launch_copy_rows(h->n, h->rl, h->Wp, h->rl, h->W, h->r));
    h->fu.gw_state = fused_state::NONE;
  }
  if (h->h_out) {
    if (packed) DN_TRY(launch_copy_rows(h->m, h->rl, h->Hp, h->rl, h->H, h->r));
    h->fu.gh_state = fused_state::NONE;
    h->gh_valid = h->nw_valid = h->fu_n_valid = false;
  }
  return 0;
}

// At the end of every call that changes a factor in place: packed copies whose pointers are out show it.
static int show(dnpeff_nmf* h, bool w, bool hh) {
  if (h->r == h->rl) return 0;
  if (w && h->w_out) DN_TRY(launch_copy_rows(h->n, h->rl, h->W, h->r, h->Wp, h->rl));
  if (hh && h->h_out) DN_TRY(launch_copy_rows(h->m, h->rl, h->H, h->r, h->Hp, h->rl));
  return 0;
}

static bool fused_now(const dnpeff_nmf* h) {
  return h->has_fused && tuning().fused_gram != 0.0 && !h->A->tail && !h->prof.enabled;
}

static bool small_now(const dnpeff_nmf* h) {
  return fused_now(h) && h->A->n_panels == 0 && has_row_major(h->A) && h->A->colptr &&
         fused_small_fits(h->n, h->m, h->A->nnz, h->r);
}

DN_API int dnpeff_nmf_destroy(dnpeff_nmf* nmf) {
  if (!nmf) return 0;
  (void)hipStreamSynchronize(stream());
  dfree(nmf->W); dfree(nmf->W2); dfree(nmf->Nw); dfree(nmf->Hbuf); dfree(nmf->S); dfree(nmf->S2);
  dfree(nmf->G); dfree(nmf->G2); dfree(nmf->gram_ws); dfree(nmf->dot_ws);
  dfree(nmf->GH); dfree(nmf->gpart); dfree(nmf->Wp); dfree(nmf->Hp);
  nmf->fu.destroy();
  delete nmf;
  return 0;
}

// The H update also produces H^T H (one pass over H instead of two) when the rank is 128 and
// the factor is large enough for the pass to matter (fused_gram switch: 0 = off).
static bool fused_update(const dnpeff_nmf* h) {
  if (tuning().fused_gram == 0.0 || h->tiled) return false;
  return h->r == 128 && h->m >= 4096;
}

// Rows that the arrays of a factor have memory for: whole tiles of the update kernel where the rank has one.
static int64_t rows_there(int r, int64_t rows) {
  return r > 128 && r % 128 == 0 ? ceil_div(rows, 128) * 128 : rows;
}

// Columns of a tile of the tiled H update: h_tile_mb MiB of the factor, a multiple of 128.
static int64_t tile_cols_for(int64_t m, int rank) {
  double mb = tuning().h_tile_mb;
  if (mb < 0.001) mb = 0.001;
  int64_t t = (int64_t)(mb * 1024.0 * 1024.0 / (4.0 * rank)) / 128 * 128;
  if (t < 128) t = 128;
  const int64_t m_pad = ceil_div(m, 128) * 128;
  return t < m_pad ? t : m_pad;
}

// Bytes of device memory that the handle allocates besides the structures of the matrix.
static double factor_bytes(int64_t n, int64_t m, int rank, int asked, bool tiled) {
  const int64_t run = rank != asked ? PADDED_GRAM_RUN : 0;
  const double nr = 4.0 * (double)n * rank, mr = 4.0 * (double)m * rank;
  const double spare = 5.0 * 4.0 * (double)(rank > 128 && rank % 128 == 0 ? 128 * rank : 4);  // (rows_there, 16-byte loads)
  const double packed = rank != asked ? 4.0 * (double)asked * (double)(n + m) : 0.0;
  double ws = (double)gram_workspace_floats(m, rank, run), ws_n = (double)gram_workspace_floats(n, rank, run);
  if (ws_n > ws) ws = ws_n;
  const double tile = 4.0 * (double)tile_cols_for(m, rank) * rank;
  return 3.0 * nr + (tiled ? mr + 2.0 * tile : 2.0 * mr) + 4.0 * ws + 3.0 * 4.0 * rank * rank +
         4.0 * (double)xg_mu_gram_workspace_floats(m) + spare + packed;
}

// What the products' own buffers take besides the two sparse copies (16 bytes per entry of the
// sparse part), the dense blocks and the head's workspace, which the choice of the head prices
// per candidate: upper bounds from the same rules that size the allocations.
struct plan_table {
  double factors = 0.0;   // W, its double buffer, A H^T, H (+ tile), A^T W (or its tile), Grams, workspaces, packed copies
  double partials = 0.0;  // partial sums of A H^T: per 2048-entry chunk, or per (row, plain panel / XCD)
  double segments = 0.0;  // offsets of the (row, panel) segments
  double offsets = 0.0;   // column offsets, long-column list, row offsets and chunk counts, tiles of A^T W
  double reserve = 0.0;   // left free (1/64 of the device, at least 1 GiB): allocation granularity, code objects, the runtime's own
  double total() const { return factors + partials + segments + offsets + reserve; }
};

// rank: as stored, asked: the caller's.
static plan_table plan_overheads(int64_t n, int64_t m, int64_t nnz_sparse, int rank, int asked, bool tiled, bool sweeps,
                                 double total_bytes) {
  plan_table t;
  t.factors = factor_bytes(n, m, rank, asked, tiled);
  const int64_t P = coarse_panels_for(n, m, rank, sweeps);
  const double by_chunks = 4.0 * rank * ((double)nnz_sparse / (double)SPMM_N_CHUNK + (double)n);
  const double by_panels = P > 0 ? 4.0 * rank * (double)n * (double)(P + SWEEP_XCDS) : 0.0;
  t.partials = by_chunks > by_panels ? by_chunks : by_panels;
  // (a coarse panel may be cut into swept pieces: up to max_panels() panels and pieces in all)
  t.segments = P > 0 ? 8.0 * (double)n * (double)((sweeps ? max_panels() : P) + 1) : 0.0;
  const double n_long = std::min((double)m, (double)nnz_sparse / (double)(SPMM_T_LONG + 1));
  t.offsets = 8.0 * (double)(m + 1) + 4.0 * n_long + 2.0 * 8.0 * (double)(n + 1) + 2.0 * 8.0 * 64.0;
  if (rank > 128) t.offsets += spmm_t_bal_fits(n, rank) ? fused_tiles_bytes(m, nnz_sparse) : 0.0;
  t.reserve = std::max(1073741824.0, total_bytes / 64.0);
  return t;
}

// Whether a rank is stored as the next multiple of 128.  At 500 x 823k ten updates take 111 ms at r = 301 as it
// is (fp32 matrix cores, 4-byte loads) and 41 ms with 384 components of which 83 are zero.  Not where the longer
// rows, with the packed copies that callers may ask for, do not fit into `there` bytes.
static int stored_rank(int64_t n, int64_t m, int64_t nnz, int rank, bool sweeps, double there, double total_bytes) {
  const int p = (rank + 127) / 128 * 128;
  if (rank <= 128 || p == rank || !use_split_bf16() || tuning().pad_rank == 0.0 || tuning().tiled_h > 0.0) return rank;
  const plan_table t = plan_overheads(n, m, nnz, p, rank, false, sweeps, total_bytes);
  return t.total() + 24.0 * (double)nnz <= there ? p : rank;
}

// Whether the step of small ranks runs where memory allows.  It reads the whole matrix from its own lists: no
// dense head is split off then.
// Rank 128 with rows enough for a dense head keeps it: the fused step's kernel at that rank has one wave per SIMD.
// Ten iterations with head / fused: 14.7 / 16.0 ms at 1500 x 1.4M, 24.2 / 31.2 at 2000 x 1.9M, 79 / 84 at 2000 x
// 9.8M, but 8.5 / 7.2 at 1024 x 0.8M.
// Rank 64 keeps it where the matrix is dense: a gathered entry takes as long as eight cells of the head, and the head's
// launches as long as 6 M entries (1.7 ms in ten iterations).  Ten iterations with head / fused, by the share of the
// cells that hold an entry: 23.3 / 40.7 ms at 2000 x 200k, 120 M entries (0.30), 3.17 / 4.49 at 1500 x 20k, 15 M (0.50),
// 3.17 / 3.50 with 12 M (0.40) but 3.17 / 2.51 with 8.3 M (0.28), 34.1 / 43.2 at 4000 x 200k (0.16), 18.7 / 20.6 at 8000 x
// 60k (0.14), 10.4 / 10.7 at 4000 x 60k (0.14) but 5.6 / 3.4 at 3000 x 20k, 12 M (0.20), 23.0 / 21.7 at 4000 x 200k
// (0.08), 57 / 53 at 20000 x 200k (0.04).  Below, the fused step is ahead by 1.1 to 5 from 1024 x 1100 to 100000 x
// 4.0M (1.73 / 0.32, 3.4 / 1.3 at 1100 x 60k, 52 / 36 at 8000 x 5.7M, 145 / 107), unless few columns hold most of very many
// entries (head_beats_fused).  It is also closer to 64 bits: one W update 5e-7 ... 8e-7 off where the head's split operands
// leave 1e-6 ... 6e-6.
static bool fused_step_wanted(int64_t n, int64_t m, int64_t nnz, int rank) {
  if (tuning().fused_gram == 0.0 || tuning().tiled_h > 0.0 || !fused_supported(n, m, nnz, rank)) return false;
  if (n < 1024 || rank % 64 != 0) return true;
  return rank == 64 && 9.0 * ((double)nnz - 6e6) <= (double)n * (double)m;
}

// Rank 64, a head of z_head entries on the columns that a sixteenth of the rows hold: it pays for its launches and the passes
// over H that the fused step does without (27 M entries and 7 to a column), and for the rest of the matrix, which its kernels
// take at half the speed.  Of 313 matrices of 16 to 330 M entries (1030 to 70,000 rows, Zipf laws of 1.05 to 1.6) the choice
// is 0.7 % from the faster way on average and 1.22 at most; by the rule for dense matrices alone 4.8 % and 1.61.  Five
// iterations with head / fused: 36.3 / 45.0 ms at 40,000 x 1.8M with 262 M entries, exponent 1.6, 39.3 / 50.7 at 2000 x 3.9M with
// 262 M, 1.3, 8.0 / 11.5 at 40,000 x 50k with 66 M, 1.6, 8.8 / 10.4 at 12,000 x 165k; past the line 13.4 / 11.4 at 12,000 x 1.1M with
// 66 M, 1.6, 10.5 / 10.5 at 12,000 x 165k, 1.3, 24.5 / 23.5 at 40,000 x 1.0M with 131 M, 1.3, 27.2 / 24.2 at 5000 x 786k, 1.05.
static bool head_beats_fused(int64_t m, int64_t nnz, int64_t z_head) {
  return (double)z_head > 27e6 + (double)(nnz - z_head) + 7.0 * (double)m;
}

// Whether it does within `budget` bytes beside the factors, and whether with lists by XCD.
struct fused_choice {
  bool on = false, xcd = false;
  double lists = 0.0, state = 0.0;  // bytes
};
static fused_choice choose_fused(int64_t n, int64_t m, int64_t nnz, int rank, double budget) {
  fused_choice c;
  if (!fused_step_wanted(n, m, nnz, rank)) return c;
  c.lists = fused_list_bytes(n, m, nnz);
  c.state = fused_state_bytes(n, m, nnz, rank);
  const double need = 16.0 * (double)nnz + c.lists + c.state, more = fused_xcd_bytes(n, nnz, rank);
  c.on = need < budget;
  c.xcd = more > 0.0 && need + more < budget;
  if (c.xcd) c.lists += more;
  return c;
}

// For tests and capacity planning without a GPU: the table above and, for a head of n_dense columns,
// its blocks and workspace.  out[0..7] = factors, partials, segments, offsets, reserve, sparse
// copies, head blocks, head workspace (bytes).
DN_API int dnpeff_plan_estimate(int64_t n_rows, int64_t n_cols, int64_t nnz_sparse, int64_t n_dense, int rank,
                                int tiled, int sweeps, int64_t total_bytes, double* out) {
  clear_error();
  DN_CHECK(out != nullptr, "out is NULL");
  DN_CHECK(n_rows >= 0 && n_cols >= 0 && nnz_sparse >= 0 && n_dense >= 0 && n_dense <= n_cols,
           "negative size");
  DN_CHECK(rank >= 1 && rank <= 1024, "rank %d outside [1, 1024]", rank);
  const double total = (double)total_bytes;
  const int asked = rank;
  if (!tiled) rank = stored_rank(n_rows, n_cols, nnz_sparse, asked, sweeps != 0, total, total);
  plan_table t = plan_overheads(n_rows, n_cols, nnz_sparse, rank, asked, tiled != 0, sweeps != 0, total);
  out[5] = 16.0 * (double)nnz_sparse;
  const fused_choice fused = choose_fused(n_rows, n_cols, nnz_sparse, rank, total - t.total());
  if (!tiled && n_dense == 0 && fused.on) {
    out[5] += fused.lists;
    t.factors += fused.state;
  }
  out[0] = t.factors; out[1] = t.partials; out[2] = t.segments; out[3] = t.offsets; out[4] = t.reserve;
  out[6] = n_dense ? 4.0 * head_blocks_for_rank(rank) * (double)(ceil_div(n_rows, 128) * 128) *
                         (double)(ceil_div(n_dense, 128) * 128)
                   : 0.0;
  out[7] = 4.0 * (double)head_workspace_floats(n_rows, n_dense, rank, head_run(rank, asked));
  return 0;
}

// Splits off the dense head when the products can use it: rank a multiple of 4 and at least 64
// (below that a column of the dense block costs more than its entries do as gathers), enough
// rows for the fill fraction to mean something.  A column goes to the head when at least 1/16 of
// the rows hold it (dense_fill switch; 0 = never split); the fraction is raised until the dense
// blocks and both sparse copies of the rest fit the memory left beside the factors.  *tiled
// receives whether the H update must run on column tiles for everything to fit.
// *fused: whether the step of small ranks runs.
static int plan_matrix(dnpeff_csr* A, int rank, int asked, bool consume, bool* tiled, fused_choice* fused) {
  const tuning_t& tn = tuning();
  size_t free_b = 0, total_b = 0;
  DN_HIP(hipMemGetInfo(&free_b, &total_b));
  const dnpeff_csr* S0 = sparse_part(A);
  // memory that the matrix structures may take: what is free now, plus what a consuming create
  // releases, plus what the structures hold already
  double avail = (double)free_b + (double)pool_cached_bytes();
  if (consume && A->colind && A->vals) avail += 8.0 * (double)A->nnz;
  if (A->tail) {
    avail += (A->head.rm ? 8.0 : 4.0) * (double)A->head.n_pad * (double)A->head.n_d_pad;
    if (S0->colind) avail += 8.0 * (double)S0->nnz;
  }
  if (S0->colptr) avail += 8.0 * (double)S0->nnz;
  if (S0->pcol || S0->nl.pairs) avail += 8.0 * (double)S0->nnz;
  const bool sweeps = sweeps_for_rank(rank);
  const plan_table t_full = plan_overheads(A->n_rows, A->n_cols, A->nnz, rank, asked, false, sweeps, (double)total_b);
  const plan_table t_tiled = plan_overheads(A->n_rows, A->n_cols, A->nnz, rank, asked, true, sweeps, (double)total_b);
  const double budget_full = avail - t_full.total();
  const double budget_tiled = avail - t_tiled.total();
  *fused = choose_fused(A->n_rows, A->n_cols, A->nnz, rank, budget_full);
  head_choice c;
  bool chosen = false;
  if (fused->on && rank == 64 && A->n_rows >= 1024 && !A->tail && has_row_major(A) && tn.dense_fill <= 1.0 &&
      head_beats_fused(A->n_cols, A->nnz, A->nnz)) {
    DN_TRY(choose_dense_head(A, tn.dense_fill, budget_full, head_blocks_for_rank(rank), rank, head_run(rank, asked), &c));
    chosen = c.thr > 0 && c.fits && head_beats_fused(A->n_cols, A->nnz, c.z_head);
    if (chosen) *fused = fused_choice();
  }
  const bool can_split = rank % 4 == 0 && rank >= 64 && A->n_rows >= 1024 && !fused->on;
  double fill = tn.dense_fill;
  if (fill > 1.0) fill = 0.0;
  *tiled = tn.tiled_h > 0.0;
  if (A->tail) {
    if (rank % 4 == 0) {  // split by the caller (or an earlier handle): keep it
      const double foot = 4.0 * head_blocks_for_rank(rank) * (double)A->head.n_pad * (double)A->head.n_d_pad +
                          16.0 * (double)S0->nnz + 4.0 * (double)head_workspace_floats(A->n_rows, A->head.n_d, rank, head_run(rank, asked));
      if (tn.tiled_h < 0.0) *tiled = foot > budget_full;
      return 0;
    }
    DN_TRY(dnpeff_csr_split_dense_head(A, 0.0, nullptr));
    fill = 0.0;
  }
  if (!can_split) fill = 0.0;
  if (!has_row_major(A)) {  // consumed by an earlier handle without a head: nothing to choose
    if (tn.tiled_h < 0.0) *tiled = 16.0 * (double)A->nnz > budget_full;
    return 0;
  }
  const int n_blocks = head_blocks_for_rank(rank);
  if (!chosen) DN_TRY(choose_dense_head(A, fill, *tiled ? budget_tiled : budget_full, n_blocks, rank, head_run(rank, asked), &c));
  if (!c.fits && tn.tiled_h < 0.0 && !*tiled) {
    *tiled = true;
    DN_TRY(choose_dense_head(A, fill, budget_tiled, n_blocks, rank, head_run(rank, asked), &c));
  }
  if (tn.verbose != 0.0) {
    const plan_table& t = *tiled ? t_tiled : t_full;
    fprintf(stderr,
            "dnpeff: plan for rank %d: %.1f GB free, budget for the matrix %.1f GB (%s H update); dense "
            "head of %lld columns (>= %lld entries), footprint %.1f GB%s\n"
            "dnpeff: plan bytes: factors %.2f GB, partial sums %.2f GB, segment offsets %.2f GB, column "
            "offsets %.2f GB, reserve %.2f GB\n",
            rank, (double)free_b / 1e9, (*tiled ? budget_tiled : budget_full) / 1e9,
            *tiled ? "tiled" : "full-size", (long long)c.n_d, (long long)c.thr, c.footprint / 1e9,
            c.fits ? "" : " (over budget)", t.factors / 1e9, t.partials / 1e9, t.segments / 1e9,
            t.offsets / 1e9, t.reserve / 1e9);
  }
  if (c.thr == 0) return 0;  // no head (there is none to undo either)
  return split_dense_head_at(A, c.thr, nullptr);
}

// The rank that the factors are stored with.  Padded ones need an eps that keeps 0 * (0 / eps) zero.
static int padded_rank(const dnpeff_csr* A, int rank, float eps, int* out) {
  *out = rank;
  if (rank <= 128 || !(eps >= 1e-30f)) return 0;
  size_t free_b = 0, total_b = 0;
  DN_HIP(hipMemGetInfo(&free_b, &total_b));
  *out = stored_rank(A->n_rows, A->n_cols, A->nnz, rank, sweeps_for_rank((rank + 127) / 128 * 128), (double)free_b + (double)pool_cached_bytes(), (double)total_b);
  return 0;
}

static int nmf_create_impl(dnpeff_csr* A, int rank, float eps, int64_t seed, unsigned flags,
                           dnpeff_nmf** out) {
  clear_error();
  DN_CHECK(out != nullptr, "out is NULL");
  *out = nullptr;
  DN_CHECK(A != nullptr, "matrix is NULL");
  DN_CHECK(rank >= 1 && rank <= 1024, "rank %d outside [1, 1024]", rank);
  DN_CHECK((flags & ~(unsigned)DNPEFF_NMF_CONSUME_MATRIX) == 0, "unknown flags 0x%x", flags);
  // multi_mu_dense_factors_nmf1.h:95-99
  DN_CHECK(A->n_rows <= A->n_cols, "Error: Not handling matrices with more rows than columns yet.");
  const bool consume = (flags & DNPEFF_NMF_CONSUME_MATRIX) != 0;
  // with verbose set: seconds of each phase of the set-up (the stream is drained at every mark)
  const bool timed = tuning().verbose != 0.0;
  auto t_last = std::chrono::steady_clock::now();
  auto mark = [&](const char* what) {
    if (!timed) return;
    (void)hipStreamSynchronize(stream());
    const auto t = std::chrono::steady_clock::now();
    fprintf(stderr, "dnpeff: set-up: %-44s %7.3f s\n", what, std::chrono::duration<double>(t - t_last).count());
    t_last = t;
  };
  double sq_norm = 0.0;
  DN_TRY(dnpeff_csr_sq_norm(A, &sq_norm));
  mark("||A||^2");
  const int rank_asked = rank;
  DN_TRY(padded_rank(A, rank_asked, eps, &rank));
  bool tiled = false;
  fused_choice fused;
  DN_TRY(plan_matrix(A, rank, rank_asked, consume, &tiled, &fused));
  if (tiled && rank != rank_asked) {  // (only where the two estimates of the memory disagree)
    rank = rank_asked;
    DN_TRY(plan_matrix(A, rank, rank_asked, consume, &tiled, &fused));
  }
  mark("memory plan, dense head and sparse tail");
  if (consume && A->tail) {  // the tail and the head hold everything the products read
    DN_HIP(hipStreamSynchronize(stream()));
    dfree(A->colind); A->colind = nullptr;
    dfree(A->vals); A->vals = nullptr;
  }
  A->head.t_run = head_run(rank, rank_asked);
  DN_TRY(csr_ensure_products(A, rank));
  mark("transposed copy, panels, pieces, work lists");
  if (consume) DN_TRY(csr_consume_for_products(A));
  mark("release of what the products do not read");
  dnpeff_nmf* h = new dnpeff_nmf();
  h->A = A; h->r = rank; h->rl = rank_asked; h->eps = eps; h->seed = (uint64_t)seed;
  h->n = A->n_rows; h->m = A->n_cols;
  h->sq_norm_A = sq_norm;
  h->tiled = tiled && A->n_cols > 0;
  h->tile_cols = h->tiled ? tile_cols_for(h->m, rank) : 0;
  const int64_t n_there = rows_there(rank, h->n), m_there = rows_there(rank, h->m);
  const int64_t nr = n_there * rank, mr = m_there * rank;
  const int64_t h_floats = h->tiled ? (m_there + h->tile_cols) * rank : mr;
  const int64_t s_floats = h->tiled ? h->tile_cols * rank : mr;
  int64_t ws = gram_workspace_floats(h->m, rank, gram_run(h));
  int64_t ws_n = gram_workspace_floats(h->n, rank, gram_run(h));
  if (ws_n > ws) ws = ws_n;
  // (four spare floats: the step of small ranks reads rows in 16-byte pieces)
  int s = dmalloc(&h->W, nr + 4) || dmalloc(&h->W2, nr + 4) || dmalloc(&h->Nw, nr + 4) ||
          dmalloc(&h->Hbuf, h_floats + 4) || dmalloc(&h->S, s_floats + 4) ||
          dmalloc(&h->G, (int64_t)rank * rank) || dmalloc(&h->G2, (int64_t)rank * rank) ||
          dmalloc(&h->gram_ws, ws) || dmalloc(&h->dot_ws, DOT_BLOCKS + 2);
  h->H = h->Hbuf;
  if (!s && fused_update(h))
    s = dmalloc(&h->GH, (int64_t)rank * rank) || dmalloc(&h->gpart, xg_mu_gram_workspace_floats(h->m));
  if (!s && h->tiled && tuning().h_overlap != 0.0) s = dmalloc(&h->S2, s_floats);
  if (!s && h->tiled) s = csr_tile_lists(A);
  if (!s && fused.on && !h->tiled && !A->tail) {
    h->has_fused = true;
    s = fused_plan_build(A, rank, fused.xcd) || h->fu.create(A, h->n, rank, fused.xcd);
  }
  if (s) { dnpeff_nmf_destroy(h); return s; }
  mark("factors and workspaces");
  if (tuning().verbose != 0.0) {
    size_t free_b = 0, total_b = 0;
    (void)hipMemGetInfo(&free_b, &total_b);
    fprintf(stderr, "dnpeff: factors allocated (%s H update%s), %.1f GB of %.1f GB left free\n",
            h->tiled ? "tiled" : "full-size", consume ? ", matrix consumed" : "", (double)free_b / 1e9,
            (double)total_b / 1e9);
  }
  *out = h;
  return 0;
}

DN_API int dnpeff_nmf_create(dnpeff_csr* A, int rank, float eps, int64_t seed, dnpeff_nmf** out) {
  return nmf_create_impl(A, rank, eps, seed, 0u, out);
}

DN_API int dnpeff_nmf_create_ex(dnpeff_csr* A, int rank, float eps, int64_t seed, unsigned flags,
                                dnpeff_nmf** out) {
  return nmf_create_impl(A, rank, eps, seed, flags, out);
}

DN_API int dnpeff_nmf_info(const dnpeff_nmf* nmf, int* tiled, int64_t* tile_cols) {
  DN_CHECK(nmf != nullptr, "handle is NULL");
  if (tiled) *tiled = nmf->tiled ? 1 : 0;
  if (tile_cols) *tile_cols = nmf->tile_cols;
  return 0;
}

DN_API int dnpeff_nmf_init_factors(dnpeff_nmf* nmf) {
  clear_error();
  DN_CHECK(nmf != nullptr, "handle is NULL");
  nmf->gh_valid = false;
  nmf->nw_valid = false;
  nmf->fu_n_valid = false;
  nmf->fu.gh_state = nmf->fu.gw_state = fused_state::NONE;
  if (nmf->r != nmf->rl) {
    DN_TRY(launch_init_uniform(0, nmf->n, nmf->rl, nmf->seed, nmf->W2));
    DN_TRY(launch_copy_rows(nmf->n, nmf->rl, nmf->W2, nmf->rl, nmf->W, nmf->r));
    DN_TRY(launch_init_uniform(1, nmf->rl, nmf->m, nmf->seed, nmf->S));
    DN_TRY(launch_copy_rows(nmf->m, nmf->rl, nmf->S, nmf->rl, nmf->H, nmf->r));
    return show(nmf, true, true);
  }
  DN_TRY(launch_init_uniform(0, nmf->n, nmf->r, nmf->seed, nmf->W));
  DN_TRY(launch_init_uniform(1, nmf->r, nmf->m, nmf->seed, nmf->H));
  return 0;
}

DN_API int dnpeff_nmf_set_factors(dnpeff_nmf* nmf, const float* W_nr, const float* H_rm) {
  clear_error();
  DN_CHECK(nmf != nullptr, "handle is NULL");
  DN_HIP(hipStreamSynchronize(stream()));
  if (W_nr) nmf->fu.gw_state = fused_state::NONE;
  DN_TRY(take_back(nmf));
  if (W_nr && nmf->r != nmf->rl) {
    DN_HIP(copy_up(nmf->W2, W_nr, sizeof(float) * nmf->n * nmf->rl));
    DN_TRY(launch_copy_rows(nmf->n, nmf->rl, nmf->W2, nmf->rl, nmf->W, nmf->r));
  } else if (W_nr) {
    DN_HIP(copy_up(nmf->W, W_nr, sizeof(float) * nmf->n * nmf->r));
  }
  if (H_rm) {
    nmf->gh_valid = false;
    nmf->nw_valid = false;
    nmf->fu_n_valid = false;
    nmf->fu.gh_state = fused_state::NONE;
    // [r, m] row-major on the host -> [m, r] on the device, through S, a column tile at a time
    // when S holds no more
    const int64_t step = nmf->tiled ? nmf->tile_cols : nmf->m;
    if (nmf->r != nmf->rl) DN_HIP(hipMemsetAsync(nmf->H, 0, sizeof(float) * nmf->m * nmf->r, stream()));
    for (int64_t c0 = 0; c0 < nmf->m; c0 += step) {
      const int64_t len = nmf->m - c0 < step ? nmf->m - c0 : step;
      if (len == nmf->m)
        DN_HIP(copy_up(nmf->S, H_rm, sizeof(float) * len * nmf->rl));
      else
        DN_HIP(hipMemcpy2D(nmf->S, sizeof(float) * len, H_rm + c0, sizeof(float) * nmf->m,
                           sizeof(float) * len, (size_t)nmf->rl, hipMemcpyHostToDevice));
      DN_TRY(launch_transpose_ld(nmf->rl, len, nmf->S, len, nmf->H + c0 * nmf->r, nmf->r));
      DN_HIP(hipStreamSynchronize(stream()));
    }
  }
  return show(nmf, W_nr != nullptr, H_rm != nullptr);
}

// The matrix may have been planned again for another rank since this handle was made (a second
// handle, a single-kernel call): make its work lists and workspaces fit this rank again.
static int products_for(dnpeff_nmf* h) {
  h->A->head.t_run = head_run(h->r, h->rl);
  DN_TRY(csr_ensure_products(h->A, h->r));
  if (h->tiled) DN_TRY(csr_tile_lists(h->A));
  return 0;
}

// A H^T by chunks (or, where the factor is large enough for column panels, as Nw), and H^T H.
static int fused_products(dnpeff_nmf* h) {
  DN_TRY(products_for(h));
  DN_TRY(fused_plan_build(h->A, h->r, h->fu.xcd));
  if (h->A->n_panels == 0 && !h->fu.n_part_fits(h->A)) h->fu_n_valid = false;  // (the lists were built again, others)
  if (h->fu.gh_state == fused_state::NONE) DN_TRY(h->fu.gram_of(h->H, h->m, true));
  if (!h->fu_n_valid) {
    if (h->A->n_panels > 0) {
      DN_TRY(launch_spmm_n(h->A, h->r, h->H));
      DN_TRY(launch_spmm_n_reduce(h->A, h->r, h->Nw));
      h->nw_valid = true;
    } else {
      DN_TRY(h->fu.product_n(h->A, h->H));
    }
    h->fu_n_valid = true;
  }
  return h->fu.sum_h();
}

static const float* fused_nw(const dnpeff_nmf* h) { return h->A->n_panels > 0 ? h->Nw : nullptr; }

static int fused_update_W(dnpeff_nmf* h) {
  DN_TRY(fused_products(h));
  return h->fu.update_w(h->A, h->n, fused_nw(h), h->W, h->eps);
}

static int fused_update_H(dnpeff_nmf* h) {
  DN_TRY(products_for(h));
  DN_TRY(fused_plan_build(h->A, h->r, h->fu.xcd));
  if (h->fu.gw_state == fused_state::NONE) DN_TRY(h->fu.gram_of(h->W, h->n, false));
  h->nw_valid = h->gh_valid = h->fu_n_valid = false;
  return h->fu.update_h(h->A, h->W, h->H, h->eps);
}

DN_API int dnpeff_nmf_update_W(dnpeff_nmf* h) {
  DN_CHECK(h != nullptr, "handle is NULL");
  DN_TRY(take_back(h));
  h->w_out = false;
  if (fused_now(h)) return fused_update_W(h);
  h->fu.gw_state = fused_state::NONE;
  dnpeff_csr* A = h->A;
  bool gram_done = false;
  if (!h->nw_valid && !h->gh_valid && tuning().gram_beside != 0.0) {
    // H^T H on the second stream, the dense head of A H^T on the library stream behind it: the
    // head's workgroups take the CUs as those of H^T H leave them, and the rest of A H^T (kernels
    // that need the whole chip) starts when both are done.  Timing: H^T H from its start to its
    // end; A H^T from the end of H^T H to the end of the head (what the head adds), then the rest.
    DN_TRY(products_for(h));
    struct guard {
      ~guard() { side_stream_route(false); }
    } g;
    DN_TRY(side_stream_begin());
    int st = h->prof.begin(DNPEFF_K_GRAM_H);
    if (!st) st = launch_gram(h->m, h->r, h->H, h->G, h->gram_ws, gram_run(h));
    if (!st) st = h->prof.next(DNPEFF_K_SPMM_N);
    DN_TRY(side_stream_end());
    DN_TRY(st);
    gram_done = true;
    DN_TRY(launch_spmm_n(A, h->r, h->H, 1));
    DN_TRY(h->prof.end());
    DN_TRY(side_stream_join());
    DN_TRY(h->prof.resume(DNPEFF_K_SPMM_N));
    DN_TRY(launch_spmm_n(A, h->r, h->H, 2));
    DN_TRY(h->prof.end());
    DN_TRY(h->prof.begin(DNPEFF_K_SPMM_N_REDUCE));
    DN_TRY(launch_spmm_n_reduce(A, h->r, h->Nw));
    DN_TRY(h->prof.end());
    h->nw_valid = true;
  }
  if (!h->nw_valid) {  // a loss evaluation since the last H update has left A H^T in Nw
    DN_TRY(products_for(h));
    DN_TRY(h->prof.begin(DNPEFF_K_SPMM_N));
    DN_TRY(launch_spmm_n(A, h->r, h->H));
    DN_TRY(h->prof.end());
    DN_TRY(h->prof.begin(DNPEFF_K_SPMM_N_REDUCE));
    DN_TRY(launch_spmm_n_reduce(A, h->r, h->Nw));
    DN_TRY(h->prof.end());
    h->nw_valid = true;
  }
  const float* Gh = h->GH;
  DN_TRY(side_stream_join());
  if (gram_done) {
    Gh = h->G;
  } else if (!h->gh_valid) {
    DN_TRY(h->prof.begin(DNPEFF_K_GRAM_H));
    DN_TRY(launch_gram(h->m, h->r, h->H, h->G, h->gram_ws, gram_run(h)));
    DN_TRY(h->prof.end());
    Gh = h->G;
  }
  DN_TRY(h->prof.begin(DNPEFF_K_XG_MU_W));
  DN_TRY(launch_xg_mu(h->n, h->r, h->W, Gh, h->Nw, h->eps, h->W2, nullptr, rows_there(h->r, h->n)));
  DN_TRY(h->prof.end());
  std::swap(h->W, h->W2);
  return 0;
}

// The H update on column tiles: A^T W of a tile into S, then the tile's update written one tile
// away from the old tile inside Hbuf.  H at the start of Hbuf: the new H goes one tile up and
// the tiles are walked from the last to the first (a new tile then lands on old tiles that were
// read already); H one tile up: the new H goes to the start, first tile first.  The tiles are
// independent of one another, so the order does not change any sum.
// The same with A^T W of tile q + 1 (library stream) running beside the update of tile q (second
// stream of the same priority), through two tile buffers.  The updates follow one another on
// their stream, so the rule about where a new tile may land holds as it does above; a product
// waits for the update that last read its buffer.  Same kernels on the same operands: same bits.
static int update_H_tiled_overlapped(dnpeff_nmf* h) {
  dnpeff_csr* A = h->A;
  const int r = h->r;
  const int64_t tile = h->tile_cols, n_tiles = ceil_div(h->m, tile);
  const bool up = h->H == h->Hbuf;
  float* Hnew = up ? h->Hbuf + tile * r : h->Hbuf;
  static hipEvent_t ev_t[2] = {nullptr, nullptr}, ev_x[2] = {nullptr, nullptr}, fork = nullptr;
  if (!fork) {
    DN_HIP(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
    for (int b = 0; b < 2; b++) {
      DN_HIP(hipEventCreateWithFlags(&ev_t[b], hipEventDisableTiming));
      DN_HIP(hipEventCreateWithFlags(&ev_x[b], hipEventDisableTiming));
    }
  }
  hipStream_t s0 = stream(), s1 = side_stream_handle();
  DN_CHECK(s1 != nullptr, "second stream");
  struct guard {  // whatever happens, the library stream is where later launches go
    ~guard() { side_stream_route(false); xg_mu_release_g(); }
  } g;
  DN_TRY(h->prof.begin(DNPEFF_K_SPMM_T));
  DN_TRY(launch_head_t_product(A, r, h->W));
  DN_TRY(h->prof.end());
  DN_TRY(xg_mu_hold_g(h->G, r, tile));
  DN_HIP(hipEventRecord(fork, s0));
  DN_HIP(hipStreamWaitEvent(s1, fork, 0));
  for (int64_t q = 0; q < n_tiles; q++) {
    const int64_t t = up ? n_tiles - 1 - q : q;
    const int64_t c0 = t * tile, c1 = c0 + tile < h->m ? c0 + tile : h->m;
    const int b = (int)(q & 1);
    float* Sb = b ? h->S2 : h->S;
    if (q >= 2) DN_HIP(hipStreamWaitEvent(s0, ev_x[b], 0));
    DN_TRY(h->prof.begin(DNPEFF_K_SPMM_T));
    DN_TRY(launch_spmm_t_tile(A, r, h->W, c0, c1, Sb));
    DN_TRY(h->prof.end());
    DN_HIP(hipEventRecord(ev_t[b], s0));
    DN_HIP(hipStreamWaitEvent(s1, ev_t[b], 0));
    side_stream_route(true);
    DN_TRY(h->prof.begin(DNPEFF_K_XG_MU_H));
    DN_TRY(launch_xg_mu(c1 - c0, r, h->H + c0 * r, h->G, Sb, h->eps, Hnew + c0 * r, nullptr, rows_there(r, c1 - c0)));
    DN_TRY(h->prof.end());
    side_stream_route(false);
    DN_HIP(hipEventRecord(ev_x[b], s1));
  }
  DN_HIP(hipStreamWaitEvent(s0, ev_x[0], 0));
  if (n_tiles > 1) DN_HIP(hipStreamWaitEvent(s0, ev_x[1], 0));
  h->H = Hnew;
  h->gh_valid = false;
  return 0;
}

static int update_H_tiled(dnpeff_nmf* h) {
  if (h->S2) return update_H_tiled_overlapped(h);
  dnpeff_csr* A = h->A;
  const int r = h->r;
  const int64_t tile = h->tile_cols, n_tiles = ceil_div(h->m, tile);
  const bool up = h->H == h->Hbuf;
  float* Hnew = up ? h->Hbuf + tile * r : h->Hbuf;
  DN_TRY(h->prof.begin(DNPEFF_K_SPMM_T));
  DN_TRY(launch_head_t_product(A, r, h->W));
  DN_TRY(h->prof.end());
  struct held_g {  // one copy of G for all tiles
    ~held_g() { xg_mu_release_g(); }
  } hold;
  DN_TRY(xg_mu_hold_g(h->G, r, tile));
  for (int64_t q = 0; q < n_tiles; q++) {
    const int64_t t = up ? n_tiles - 1 - q : q;
    const int64_t c0 = t * tile, c1 = c0 + tile < h->m ? c0 + tile : h->m;
    // (one event per change of class: a tile's product starts where the tile before ended)
    DN_TRY(q == 0 ? h->prof.begin(DNPEFF_K_SPMM_T) : h->prof.next(DNPEFF_K_SPMM_T));
    DN_TRY(launch_spmm_t_tile(A, r, h->W, c0, c1, h->S));
    DN_TRY(h->prof.next(DNPEFF_K_XG_MU_H));
    DN_TRY(launch_xg_mu(c1 - c0, r, h->H + c0 * r, h->G, h->S, h->eps, Hnew + c0 * r, nullptr, rows_there(r, c1 - c0)));
  }
  DN_TRY(h->prof.end());
  h->H = Hnew;
  h->gh_valid = false;
  return 0;
}

DN_API int dnpeff_nmf_update_H(dnpeff_nmf* h) {
  DN_CHECK(h != nullptr, "handle is NULL");
  DN_TRY(take_back(h));
  h->h_out = false;
  if (fused_now(h)) return fused_update_H(h);
  h->fu.gh_state = fused_state::NONE;
  h->fu_n_valid = false;
  dnpeff_csr* A = h->A;
  DN_TRY(products_for(h));
  DN_TRY(h->prof.begin(DNPEFF_K_GRAM_W));
  DN_TRY(launch_gram(h->n, h->r, h->W, h->G, h->gram_ws, gram_run(h)));
  DN_TRY(h->prof.end());
  h->nw_valid = false;
  if (h->tiled) return update_H_tiled(h);
  DN_TRY(h->prof.begin(DNPEFF_K_SPMM_T));
  DN_TRY(launch_spmm_t(A, h->r, h->W, h->S));
  DN_TRY(h->prof.end());
  DN_TRY(h->prof.begin(DNPEFF_K_XG_MU_H));
  if (h->GH && ((uintptr_t)h->H % 16) == 0) {
    DN_TRY(launch_xg_mu_gram(h->m, h->H, h->G, h->S, h->eps, h->S, h->GH, h->gpart, h->G2, h->gram_ws));
    h->gh_valid = true;
  } else {
    DN_TRY(launch_xg_mu(h->m, h->r, h->H, h->G, h->S, h->eps, h->S, nullptr, rows_there(h->r, h->m)));
    h->gh_valid = false;
  }
  DN_TRY(h->prof.end());
  std::swap(h->H, h->S);
  h->Hbuf = h->H;
  return 0;
}

static int small_steps(dnpeff_nmf* nmf, int n_steps, double* sums) {
  DN_TRY(take_back(nmf));
  nmf->w_out = nmf->h_out = false;
  nmf->fu.gh_state = nmf->fu.gw_state = fused_state::NONE;
  nmf->gh_valid = nmf->nw_valid = nmf->fu_n_valid = false;
  return fused_small_launch(nmf->A, nmf->r, nmf->W, nmf->H, nmf->eps, n_steps, sums);
}

DN_API int dnpeff_nmf_step(dnpeff_nmf* nmf, int n_steps) {
  clear_error();
  DN_CHECK(nmf != nullptr, "handle is NULL");
  if (n_steps > 0 && small_now(nmf)) return small_steps(nmf, n_steps, nullptr);
  for (int s = 0; s < n_steps; s++) {
    DN_TRY(dnpeff_nmf_update_W(nmf));
    DN_TRY(dnpeff_nmf_update_H(nmf));
  }
  return 0;
}

DN_API int dnpeff_nmf_loss_terms(dnpeff_nmf* h, double* sq_norm_A, double* pos, double* neg) {
  clear_error();
  DN_CHECK(h != nullptr, "handle is NULL");
  DN_TRY(take_back(h));
  dnpeff_csr* A = h->A;
  if (fused_now(h)) {
    unsigned long long* words = nullptr;
    DN_TRY(host_words(&words));
    double* sums = reinterpret_cast<double*>(words);
    if (small_now(h)) {
      DN_TRY(fused_small_launch(A, h->r, h->W, h->H, h->eps, 0, sums));
    } else {
      DN_TRY(fused_products(h));
      if (h->fu.gw_state == fused_state::NONE) DN_TRY(h->fu.gram_of(h->W, h->n, false));
      DN_TRY(h->fu.loss_sums(A, h->n, fused_nw(h), h->W, sums));
    }
    DN_HIP(hipStreamSynchronize(stream()));
    if (sq_norm_A) *sq_norm_A = h->sq_norm_A;
    if (neg) *neg = sums[0];
    if (pos) *pos = sums[1];
    return 0;
  }
  // neg = <W^T A, H> = <A H^T, W>
  if (!h->nw_valid) {
    DN_TRY(products_for(h));
    DN_TRY(launch_spmm_n(A, h->r, h->H));
    DN_TRY(launch_spmm_n_reduce(A, h->r, h->Nw));
    h->nw_valid = true;
  }
  DN_TRY(launch_dot(h->n * h->r, h->Nw, h->W, h->dot_ws, h->dot_ws + DOT_BLOCKS));
  // pos = <H, (W^T W) H> = <W^T W, H H^T>
  // (H^T H of the current H is at hand when the last H update produced it)
  const float* Gh = h->G;
  if (h->GH && h->gh_valid)
    Gh = h->GH;
  else
    DN_TRY(launch_gram(h->m, h->r, h->H, h->G, h->gram_ws, gram_run(h)));
  DN_TRY(launch_gram(h->n, h->r, h->W, h->G2, h->gram_ws, gram_run(h)));
  DN_TRY(launch_dot((int64_t)h->r * h->r, Gh, h->G2, h->dot_ws, h->dot_ws + DOT_BLOCKS + 1));
  double res[2];
  DN_HIP(hipStreamSynchronize(stream()));
  DN_HIP(copy_down(res, h->dot_ws + DOT_BLOCKS, sizeof(double) * 2));
  if (sq_norm_A) *sq_norm_A = h->sq_norm_A;
  if (neg) *neg = res[0];
  if (pos) *pos = res[1];
  return 0;
}

DN_API int dnpeff_nmf_check_products(dnpeff_nmf* h, double* via_rows, double* via_columns) {
  clear_error();
  DN_CHECK(h && via_rows && via_columns, "NULL argument");
  DN_TRY(take_back(h));
  dnpeff_csr* A = h->A;
  DN_TRY(products_for(h));
  // <A H^T, W> through the row-ordered structures
  DN_TRY(launch_spmm_n(A, h->r, h->H));
  DN_TRY(launch_spmm_n_reduce(A, h->r, h->Nw));
  h->nw_valid = true;
  DN_TRY(launch_dot(h->n * h->r, h->Nw, h->W, h->dot_ws, h->dot_ws + DOT_BLOCKS));
  DN_HIP(hipStreamSynchronize(stream()));
  DN_HIP(copy_down(via_rows, h->dot_ws + DOT_BLOCKS, sizeof(double)));
  // <A^T W, H> through the column-ordered ones (S is free between two H updates)
  double sum = 0.0;
  const int64_t step = h->tiled ? h->tile_cols : h->m;
  if (h->tiled) DN_TRY(launch_head_t_product(A, h->r, h->W));
  for (int64_t c0 = 0; c0 < h->m; c0 += step) {
    const int64_t c1 = c0 + step < h->m ? c0 + step : h->m;
    if (h->tiled)
      DN_TRY(launch_spmm_t_tile(A, h->r, h->W, c0, c1, h->S));
    else
      DN_TRY(launch_spmm_t(A, h->r, h->W, h->S));
    DN_TRY(launch_dot((c1 - c0) * h->r, h->S, h->H + c0 * h->r, h->dot_ws, h->dot_ws + DOT_BLOCKS + 1));
    double part = 0.0;
    DN_HIP(hipStreamSynchronize(stream()));
    DN_HIP(copy_down(&part, h->dot_ws + DOT_BLOCKS + 1, sizeof(double)));
    sum += part;
  }
  *via_columns = sum;
  return 0;
}

// Ticks of wall_clock64() to milliseconds.
static int ticks_to_ms(double ticks, double* ms) {
  int dev = 0, khz = 0;
  DN_HIP(hipGetDevice(&dev));
  DN_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
  *ms = khz > 0 ? ticks / (double)khz : 0.0;
  return 0;
}

namespace dn {
__global__ void __launch_bounds__(64) k_stamp(unsigned long long* out) {
  if (threadIdx.x == 0) *out = (unsigned long long)wall_clock64();
}
}  // namespace dn

// steps(), then loss(), which waits for the stream; the steps lie between two stamps of the device's clock.  (The host's clock
// asks for a wait in between: the four launches of a loss of the fused step then start on an idle device, one by one.  Ten
// iterations at 512 x 431 k, r = 16, and a loss: 547 us, 552 with the wait.)
template <class Steps, class Loss>
static int steps_then_loss(Steps steps, Loss loss, double* ms) {
  unsigned long long* stamps = nullptr;
  DN_TRY(host_stamps(&stamps));
  hipLaunchKernelGGL(k_stamp, dim3(1), dim3(64), 0, stream(), stamps);
  DN_TRY(steps());
  hipLaunchKernelGGL(k_stamp, dim3(1), dim3(64), 0, stream(), stamps + 1);
  DN_LAUNCH_CHECK();
  DN_TRY(loss());
  return ticks_to_ms((double)(stamps[1] - stamps[0]), ms);
}

DN_API int dnpeff_nmf_step_loss(dnpeff_nmf* h, int n_steps, double* loss, double* steps_ms) {
  clear_error();
  DN_CHECK(h && loss && steps_ms, "NULL argument");
  if (n_steps < 1 || n_steps > FUSED_SMALL_STEPS || !small_now(h))
    return steps_then_loss([&] { return dnpeff_nmf_step(h, n_steps); }, [&] { return dnpeff_nmf_loss(h, loss); }, steps_ms);
  unsigned long long* words = nullptr;
  DN_TRY(host_words(&words));
  double* sums = reinterpret_cast<double*>(words);
  DN_TRY(small_steps(h, n_steps, sums));
  DN_HIP(hipStreamSynchronize(stream()));
  *loss = std::sqrt(h->sq_norm_A + sums[1] - 2.0 * sums[0]);
  return ticks_to_ms(sums[2], steps_ms);
}

DN_API int dnpeff_nmf_loss(dnpeff_nmf* nmf, double* out) {
  DN_CHECK(out != nullptr, "out is NULL");
  double a, p, q;
  DN_TRY(dnpeff_nmf_loss_terms(nmf, &a, &p, &q));
  *out = std::sqrt(a + p - 2.0 * q);
  return 0;
}

DN_API int dnpeff_nmf_sparsify_W(dnpeff_nmf* nmf, float l1_norm, float l2_norm, int* rounds) {
  clear_error();
  DN_CHECK(nmf, "NULL argument");
  // (H^T H and A H^T kept between calls depend on H only)
  nmf->fu.gw_state = fused_state::NONE;
  DN_TRY(take_back(nmf));
  if (nmf->r != nmf->rl) {
    DN_TRY(launch_copy_rows(nmf->n, nmf->rl, nmf->W, nmf->r, nmf->W2, nmf->rl));
    DN_TRY(sparsify_columns(nmf->n, nmf->rl, nmf->W2, l1_norm, l2_norm, rounds));
    DN_TRY(launch_copy_rows(nmf->n, nmf->rl, nmf->W2, nmf->rl, nmf->W, nmf->r));
    return show(nmf, true, false);
  }
  return sparsify_columns(nmf->n, nmf->r, nmf->W, l1_norm, l2_norm, rounds);
}

DN_API int dnpeff_nmf_get_W(dnpeff_nmf* nmf, float* W_nr) {
  clear_error();
  DN_CHECK(nmf && W_nr, "NULL argument");
  DN_TRY(take_back(nmf));
  const float* W = nmf->W;
  if (nmf->r != nmf->rl) {
    DN_TRY(launch_copy_rows(nmf->n, nmf->rl, nmf->W, nmf->r, nmf->W2, nmf->rl));
    W = nmf->W2;
  }
  DN_HIP(hipStreamSynchronize(stream()));
  DN_HIP(copy_down(W_nr, W, sizeof(float) * nmf->n * nmf->rl));
  return 0;
}

DN_API int dnpeff_nmf_get_H(dnpeff_nmf* nmf, float* H_rm) {
  clear_error();
  DN_CHECK(nmf && H_rm, "NULL argument");
  DN_TRY(take_back(nmf));
  // [m, r] on the device -> [r, m] row-major on the host, through S: all at once, or a column
  // tile at a time when S holds no more (the tiled H update)
  const int64_t step = nmf->tiled ? nmf->tile_cols : nmf->m;
  for (int64_t c0 = 0; c0 < nmf->m; c0 += step) {
    const int64_t len = nmf->m - c0 < step ? nmf->m - c0 : step;
    DN_TRY(launch_transpose_ld(len, nmf->rl, nmf->H + c0 * nmf->r, nmf->r, nmf->S, len));
    DN_HIP(hipStreamSynchronize(stream()));
    if (len == nmf->m)
      DN_HIP(copy_down(H_rm, nmf->S, sizeof(float) * len * nmf->rl));
    else
      DN_HIP(hipMemcpy2D(H_rm + c0, sizeof(float) * nmf->m, nmf->S, sizeof(float) * len,
                         sizeof(float) * len, (size_t)nmf->rl, hipMemcpyDeviceToHost));
  }
  return 0;
}

DN_API int dnpeff_nmf_device_factors(dnpeff_nmf* nmf, void** W_dev, void** H_dev) {
  DN_CHECK(nmf != nullptr, "handle is NULL");
  const bool packed = nmf->r != nmf->rl;
  if (packed && W_dev && !nmf->w_out) {
    if (!nmf->Wp) DN_TRY(dmalloc(&nmf->Wp, nmf->n * nmf->rl));
    DN_TRY(launch_copy_rows(nmf->n, nmf->rl, nmf->W, nmf->r, nmf->Wp, nmf->rl));
  }
  if (packed && H_dev && !nmf->h_out) {
    if (!nmf->Hp) DN_TRY(dmalloc(&nmf->Hp, nmf->m * nmf->rl));
    DN_TRY(launch_copy_rows(nmf->m, nmf->rl, nmf->H, nmf->r, nmf->Hp, nmf->rl));
  }
  if (W_dev) *W_dev = packed ? nmf->Wp : nmf->W;
  if (H_dev) *H_dev = packed ? nmf->Hp : nmf->H;
  nmf->w_out = nmf->w_out || W_dev;
  nmf->h_out = nmf->h_out || H_dev;
  return 0;
}

DN_API int dnpeff_nmf_set_profiling(dnpeff_nmf* nmf, int enable) {
  DN_CHECK(nmf != nullptr, "handle is NULL");
  DN_TRY(nmf->prof.collect());
  nmf->prof.enabled = enable != 0;
  return 0;
}

DN_API int dnpeff_nmf_timings(dnpeff_nmf* nmf, double* ms_sum, int64_t* launches, int reset) {
  DN_CHECK(nmf != nullptr, "handle is NULL");
  DN_TRY(nmf->prof.collect());
  for (int i = 0; i < DNPEFF_K_COUNT; i++) {
    if (ms_sum) ms_sum[i] = nmf->prof.ms_sum[i];
    if (launches) launches[i] = nmf->prof.launches[i];
  }
  if (reset) nmf->prof.reset();
  return 0;
}

// ---------------------------------------------------------------------------
// Fixed sparse H, W-only learner
// ---------------------------------------------------------------------------
struct dnpeff_fit {
  int64_t n = 0;
  int r = 0;
  float eps = 0.0f;
  uint64_t seed = 0;
  float* AH = nullptr;   // [n, r]
  float* HH = nullptr;   // [r, r]
  float* W = nullptr;    // [n, r]
  bool in_place = false; // all steps of a call in one launch (fit.hip), without the two buffers below
  float* W2 = nullptr;   // [n, r]
  float* WHH = nullptr;  // [n, r] W (H H^T) of the W before the last step
  float* tmp = nullptr;  // [n, r]
  double* dot_ws = nullptr;
  double sq_norm_A = 0.0;
  bool whh_valid = false;
};

DN_API int dnpeff_fit_destroy(dnpeff_fit* f) {
  if (!f) return 0;
  (void)hipStreamSynchronize(stream());
  dfree(f->AH); dfree(f->HH); dfree(f->W); dfree(f->W2); dfree(f->WHH); dfree(f->tmp);
  dfree(f->dot_ws);
  delete f;
  return 0;
}

DN_API int dnpeff_fit_create(dnpeff_csr* A, dnpeff_csr* H, float eps, int64_t seed,
                             dnpeff_fit** out) {
  clear_error();
  DN_CHECK(out != nullptr, "out is NULL");
  *out = nullptr;
  DN_CHECK(A && H, "matrix is NULL");
  DN_CHECK(A->n_cols == H->n_cols, "A has %lld columns but H has %lld", (long long)A->n_cols,
           (long long)H->n_cols);
  const int r = (int)H->n_rows;
  DN_CHECK(r >= 1 && r <= 1024, "rank %d outside [1, 1024]", r);
  dnpeff_fit* f = new dnpeff_fit();
  f->n = A->n_rows; f->r = r; f->eps = eps; f->seed = (uint64_t)seed;
  const int64_t nr = f->n * r;
  f->in_place = fit_steps_supported(f->n, r);
  int64_t dots = DOT_BLOCKS + 2;
  if (f->in_place && 3 * fit_loss_parts(f->n) > dots) dots = 3 * fit_loss_parts(f->n);
  int s = dmalloc(&f->AH, nr) || dmalloc(&f->HH, (int64_t)r * r) || dmalloc(&f->W, nr) ||
          dmalloc(&f->WHH, nr) || dmalloc(&f->dot_ws, dots);
  if (!s && !f->in_place) s = dmalloc(&f->W2, nr) || dmalloc(&f->tmp, nr);
  if (!s) s = spsp_first_stage(A, H, f->HH, f->AH);
  if (!s) s = dnpeff_csr_sq_norm(A, &f->sq_norm_A);  // (the first stage is not waited for: the steps follow it on the stream)
  if (s) { dnpeff_fit_destroy(f); return s; }
  *out = f;
  return 0;
}

DN_API int dnpeff_fit_init_W(dnpeff_fit* f) {
  clear_error();
  DN_CHECK(f != nullptr, "handle is NULL");
  f->whh_valid = false;
  return launch_init_uniform(0, f->n, f->r, f->seed, f->W);
}

DN_API int dnpeff_fit_set_W(dnpeff_fit* f, const float* W_nr) {
  clear_error();
  DN_CHECK(f && W_nr, "NULL argument");
  DN_HIP(hipStreamSynchronize(stream()));
  DN_HIP(copy_up(f->W, W_nr, sizeof(float) * f->n * f->r));
  f->whh_valid = false;
  return 0;
}

DN_API int dnpeff_fit_step(dnpeff_fit* f, int n_steps) {
  clear_error();
  DN_CHECK(f != nullptr, "handle is NULL");
  if (n_steps <= 0) return 0;
  if (f->in_place) {
    f->whh_valid = true;
    return launch_fit_steps(f->n, f->r, f->W, f->HH, f->AH, f->eps, n_steps, f->WHH, nullptr);
  }
  struct held_g {  // H H^T is the same in every step: one copy for all of them
    ~held_g() { xg_mu_release_g(); }
  } hold;
  DN_TRY(xg_mu_hold_g(f->HH, f->r, f->n));
  for (int s = 0; s < n_steps; s++) {
    DN_TRY(launch_xg_mu(f->n, f->r, f->W, f->HH, f->AH, f->eps, f->W2, f->WHH));
    std::swap(f->W, f->W2);
    f->whh_valid = true;
  }
  return 0;
}

DN_API int dnpeff_fit_loss(dnpeff_fit* f, double* reference_loss, double* true_loss) {
  clear_error();
  DN_CHECK(f != nullptr, "handle is NULL");
  const int64_t nr = f->n * f->r;
  if (f->in_place) {
    unsigned long long* words = nullptr;
    DN_TRY(host_words(&words));
    double* out = reinterpret_cast<double*>(words);
    const int64_t parts = fit_loss_parts(f->n);
    const bool here = 3 * parts <= HOST_WORDS;  // (the workgroups' sums, added up here in order)
    DN_TRY(launch_fit_loss(f->n, f->r, f->W, f->HH, f->AH, f->whh_valid ? f->WHH : nullptr, here ? out : f->dot_ws,
                           here ? nullptr : out));
    DN_HIP(hipStreamSynchronize(stream()));
    double sums[3] = {out[0], out[1], out[2]};
    for (int64_t q = 3; here && q < 3 * parts; q++) sums[q % 3] += out[q];
    const double pos_ref = f->whh_valid ? sums[2] : sums[1];
    if (true_loss) *true_loss = std::sqrt(f->sq_norm_A + sums[1] - 2.0 * sums[0]);
    if (reference_loss) *reference_loss = std::sqrt(f->sq_norm_A + pos_ref - 2.0 * sums[0]);
    return 0;
  }
  double res[2];
  // neg = <A H^T, W>
  DN_TRY(launch_dot(nr, f->AH, f->W, f->dot_ws, f->dot_ws + DOT_BLOCKS));
  // pos of the current W; W2 receives an update that is discarded
  DN_TRY(launch_xg_mu(f->n, f->r, f->W, f->HH, f->AH, f->eps, f->W2, f->tmp));
  DN_TRY(launch_dot(nr, f->tmp, f->W, f->dot_ws, f->dot_ws + DOT_BLOCKS + 1));
  DN_HIP(hipStreamSynchronize(stream()));
  DN_HIP(copy_down(res, f->dot_ws + DOT_BLOCKS, sizeof(double) * 2));
  const double neg = res[0], pos_true = res[1];
  if (true_loss) *true_loss = std::sqrt(f->sq_norm_A + pos_true - 2.0 * neg);
  if (reference_loss) {
    double pos_ref = pos_true;
    if (f->whh_valid) {
      DN_TRY(launch_dot(nr, f->WHH, f->W, f->dot_ws, f->dot_ws + DOT_BLOCKS));
      DN_HIP(hipStreamSynchronize(stream()));
      DN_HIP(copy_down(&pos_ref, f->dot_ws + DOT_BLOCKS, sizeof(double)));
    }
    *reference_loss = std::sqrt(f->sq_norm_A + pos_ref - 2.0 * neg);
  }
  return 0;
}

DN_API int dnpeff_fit_step_loss(dnpeff_fit* f, int n_steps, double* reference_loss, double* true_loss, double* steps_ms) {
  clear_error();
  DN_CHECK(f && steps_ms, "NULL argument");
  if (!f->in_place || !fit_loss_with_steps(f->n, n_steps))
    return steps_then_loss([&] { return dnpeff_fit_step(f, n_steps); },
                           [&] { return dnpeff_fit_loss(f, reference_loss, true_loss); }, steps_ms);
  unsigned long long* words = nullptr;
  DN_TRY(host_words(&words));
  const double* out = reinterpret_cast<double*>(words);
  f->whh_valid = true;
  DN_TRY(launch_fit_steps(f->n, f->r, f->W, f->HH, f->AH, f->eps, n_steps, f->WHH, reinterpret_cast<double*>(words)));
  DN_HIP(hipStreamSynchronize(stream()));
  double sums[3] = {out[0], out[1], out[2]}, ticks = out[3];
  for (int64_t q = 1; q < fit_loss_parts(f->n); q++) {
    for (int k = 0; k < 3; k++) sums[k] += out[4 * q + k];
    ticks = std::max(ticks, out[4 * q + 3]);
  }
  if (true_loss) *true_loss = std::sqrt(f->sq_norm_A + sums[1] - 2.0 * sums[0]);
  if (reference_loss) *reference_loss = std::sqrt(f->sq_norm_A + sums[2] - 2.0 * sums[0]);
  return ticks_to_ms(ticks, steps_ms);
}

DN_API int dnpeff_fit_get_W(dnpeff_fit* f, float* W_nr) {
  clear_error();
  DN_CHECK(f && W_nr, "NULL argument");
  DN_HIP(hipStreamSynchronize(stream()));
  DN_HIP(copy_down(W_nr, f->W, sizeof(float) * f->n * f->r));
  return 0;
}

DN_API int dnpeff_fit_get_products(dnpeff_fit* f, float* AH_nr, float* HH_rr, double* sq_norm_A) {
  clear_error();
  DN_CHECK(f != nullptr, "handle is NULL");
  DN_HIP(hipStreamSynchronize(stream()));
  if (AH_nr) DN_HIP(copy_down(AH_nr, f->AH, sizeof(float) * f->n * f->r));
  if (HH_rr)
    DN_HIP(copy_down(HH_rr, f->HH, sizeof(float) * f->r * f->r));
  if (sq_norm_A) *sq_norm_A = f->sq_norm_A;
  return 0;
}
