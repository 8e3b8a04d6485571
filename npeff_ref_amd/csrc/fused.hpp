// The factorisation step of small ranks (fused.hip).
#pragma once

#include "dnpeff_internal.hpp"
#include "quotient.hpp"
#include "split_bf16.hpp"

#include <type_traits>

namespace dn {

constexpr int FUSED_MAX_RANK = 128;
constexpr int FUSED_NARROW_RANK = 64;  // above: fused_wide.hip
constexpr int FUW_COLS = 32;           // columns (rows of W) per tile there
// Columns whose X^T X a workgroup of the H update adds up in fp32 before it leaves the sum as a partial matrix
// (those are summed in fp64): a column with large entries takes bits from all that is added after it.  Above
// 64 components half of them where that takes no more than two rounds of workgroups.
constexpr int FU_MOST_COLS = 2048;
constexpr int FU_XCD_RANK = 96;        // ranks up to which, and entries of a row from which, A H^T goes by XCD
constexpr int64_t FU_XCD_ROW = 1792;
constexpr int64_t FU_XCD_ROW_FEW = 2560;  // (up to 8 components)
constexpr int64_t FU_CHUNKS = 4096;  // workgroups that A H^T is cut into where its rows allow

bool fused_supported(int64_t n, int64_t m, int64_t nnz, int r);
// What the lists of a matrix (alone: its tiles, which ranks above 128 use as well) and a context's buffers take at
// most, in bytes; fused_xcd_bytes: what they take on top where A H^T goes by XCD, which the step can do without.
double fused_tiles_bytes(int64_t m, int64_t nnz);
double fused_list_bytes(int64_t n, int64_t m, int64_t nnz);
double fused_xcd_bytes(int64_t n, int64_t nnz, int r);
double fused_state_bytes(int64_t n, int64_t m, int64_t nnz, int r);
// Tiles, packed entries and chunks of a matrix without dense head (needs csr_ensure_products).  xcd: the lists by XCD
// as well where its rows suit them (there is room for fused_xcd_bytes).
int fused_plan_build(dnpeff_csr* S, int r, bool xcd);

// Updates at ranks 65 ... 128 (fused_wide.hip).
int fuw_per_cu(int r, int* wgs);
int fuw_launch_h(int wgs, const fused_plan& f, const int64_t* colptr, int r, const float* W, float* H, float eps,
                 const float* gw, int n_gw, float* gpart);
int fuw_launch_w(int wgs, int64_t n, int r, const int* n_base, const float* N, float* W, float eps, const float* gh,
                 float* gpart);

// Whole runs in one workgroup's LDS (fused_small.hip): steps, then (loss: pinned, or NULL) the two sums of the loss
// and the ticks of wall_clock64() that the steps took; FUSED_SMALL_STEPS at most where these are asked for.
constexpr int FUSED_SMALL_STEPS = 1024;
bool fused_small_fits(int64_t n, int64_t m, int64_t nnz, int r);
int fused_small_launch(const dnpeff_csr* S, int r, float* W, float* H, float eps, int steps, double* loss);

// What a context keeps between the launches of a step.
struct fused_state {
  enum gram_state { NONE, PARTS, SUMMED };
  int r = 0, S_floats = 0, h_wgs = 0, w_wgs = 0;
  bool h_totals = false;     // the H update adds its Gram sums up in fp64
  bool xcd = false;          // A H^T goes by XCD where the matrix has the lists for it
  bool n_by_xcd = false;     // n_part is by XCD
  float* gh_part = nullptr;  // partial H^T H of the last H update, one per workgroup
  float* gw_part = nullptr;
  float* gh_sum = nullptr;
  float* gw_sum = nullptr;
  float* n_part = nullptr;   // A H^T by chunks
  int64_t n_part_floats = 0;
  double* dots = nullptr;
  gram_state gh_state = NONE, gw_state = NONE;

  int create(const dnpeff_csr* S, int64_t n, int rank, bool xcd_lists);
  void destroy();
  // X^T X of a factor as it is ([rows, r]): partial matrices of H or of W
  int gram_of(const float* X, int64_t rows, bool of_h);
  int product_n(const dnpeff_csr* S, const float* H);
  // whether n_part is laid out as the lists that the matrix has now say
  bool n_part_fits(const dnpeff_csr* S) const;
  int sum_h();
  int sum_w();
  // Nw: A H^T [n, r], or NULL for the chunk sums of product_n
  int update_w(const dnpeff_csr* S, int64_t n, const float* Nw, float* W, float eps);
  int update_h(const dnpeff_csr* S, const float* W, float* H, float eps);
  // out2 (device or pinned) = <A H^T, W>, <W^T W, H^T H>
  int loss_sums(const dnpeff_csr* S, int64_t n, const float* Nw, const float* W, double* out2);
};

// ---- device parts that both kernel families use ----
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int FU_GROUP = 256;        // columns whose entries are packed with one base
constexpr int FU_ROW_BITS = 24;      // a packed entry: row below, column within its 256 above
constexpr int FU_U = 4;              // gathers in flight per lane group of A H^T
constexpr int FU_U_H = 2;            // the same in the H update, where a lane takes two pieces of a row
__host__ __device__ constexpr int fu_pairs(int nb) { return nb * (nb + 1) / 2; }
__device__ inline int fu_pair(int b1, int b2, int nb) { return b1 * nb - b1 * (b1 - 1) / 2 + (b2 - b1); }

// Tile `t` of the work list (past the end: the last one), its entries cut into NG shares.
struct fu_tile_at {
  int64_t e0;
  int col0, nc, E, share;
};
template <int NG>
__device__ inline fu_tile_at fu_describe(const fu_tile* __restrict__ tiles, int n_tiles, int t) {
  fu_tile_at d;
  if (t >= n_tiles) t = n_tiles - 1;
  d.e0 = tiles[t].e0;
  d.col0 = tiles[t].col0;
  d.nc = tiles[t].cols;
  d.E = (int)(tiles[t + 1].e0 - d.e0);
  d.share = (d.E + NG - 1) / NG;
  return d;
}

// A^T W of a tile's columns into LDS, tile[column][TS], by lane groups of LPR lanes that take equal
// shares of the tile's entries.  A lane holds components 4 sub .. and 4 (sub + LPR) .. of a row.  A
// column's first part is stored to the tile, parts of later shares to carry[share][8 LPR] at CARRY.
// U gathered rows per lane group are in flight.
template <int TC, int TS, int NB, int LPR, int U = FU_U_H>
struct fu_gather {
  static constexpr int NG = 256 / LPR, CARRY = TC * TS;
  static constexpr bool WHOLE = 8 * LPR <= 16 * NB;  // both pieces of a lane lie within the padded row
  int grp, sub;
  unsigned r4, off0, off1;
  uint2 pr[U];
  unsigned before;

  __device__ inline void init(int r) {
    grp = threadIdx.x / LPR;
    sub = threadIdx.x % LPR;
    r4 = 4u * (unsigned)r;  // (pieces past the rank: any valid address)
    off0 = 4 * sub < r ? 16u * (unsigned)sub : 0u;
    off1 = 4 * (sub + LPR) < r ? 16u * (unsigned)(sub + LPR) : 0u;
  }
  // the first pairs of the group's share
  __device__ inline void request(const uint2* pairs, const fu_tile_at& d) {
    const uint2* pp = pairs + d.e0;
    const int s0 = grp * d.share;
    const unsigned last = d.E > 0 ? (unsigned)(d.E - 1) : 0u;  // (the array has a spare entry)
    before = pp[s0 > 0 && (unsigned)s0 <= last ? (unsigned)(s0 - 1) : 0u].x;
    const unsigned end = (unsigned)(s0 + d.share - 1) < last ? (unsigned)(s0 + d.share - 1) : last;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const unsigned e = (unsigned)(s0 + u);
      pr[u] = pp[e < end ? e : end];
    }
  }
  // RUN > 0: no more than RUN entries are added up one after the other before their sum joins the column's.
  template <int RUN>
  __device__ inline void run(const uint2* pairs, const fu_tile_at& d, const char* Wb, float* tile) {
    const int s0 = grp * d.share, s1 = s0 + d.share < d.E ? s0 + d.share : d.E;
    if (s0 >= s1) return;
    const uint2* pp = pairs + d.e0;
    unsigned cur = pr[0].x;
    int dst = s0 > 0 && ((cur ^ before) >> FU_ROW_BITS) == 0 ? CARRY + grp * (8 * LPR)
                                                             : (int)((cur >> FU_ROW_BITS) & (TC - 1)) * TS;
    dst += 4 * sub;
    f32x4 a0 = f32x4{0.0f, 0.0f, 0.0f, 0.0f}, a1 = a0;
    bool more = false;  // (RUN > 0) dst holds a sum of the column's entries before these
    auto put = [&]() {
      if constexpr (RUN > 0) {
        if (more) {
          a0 += *reinterpret_cast<f32x4*>(tile + dst);
          if (WHOLE || 4 * (sub + LPR) < 16 * NB) a1 += *reinterpret_cast<f32x4*>(tile + dst + 4 * LPR);
        }
      }
      *reinterpret_cast<f32x4*>(tile + dst) = a0;
      if (WHOLE || 4 * (sub + LPR) < 16 * NB) *reinterpret_cast<f32x4*>(tile + dst + 4 * LPR) = a1;
    };
#pragma unroll 1
    for (int b = s0; b < s1; b += U) {
      if constexpr (RUN > 0) {
        if (b > s0 && (b - s0) % RUN == 0) {
          put();
          more = true;
          a0 = a1 = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
      f32x4 w0[U], w1[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const unsigned at = __umul24(pr[u].x & ((1u << FU_ROW_BITS) - 1u), r4);
        w0[u] = *reinterpret_cast<const f32x4u*>(Wb + (at + off0));
        w1[u] = *reinterpret_cast<const f32x4u*>(Wb + (at + off1));
      }
      uint2 nx[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const unsigned e = (unsigned)(b + U + u), end = (unsigned)(s1 - 1);
        nx[u] = pp[e < end ? e : end];
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const float v = b + u < s1 ? __uint_as_float(pr[u].y) : 0.0f;
        if (((pr[u].x ^ cur) >> FU_ROW_BITS) != 0) {
          put();
          more = false;
          cur = pr[u].x;
          dst = (int)((cur >> FU_ROW_BITS) & (TC - 1)) * TS + 4 * sub;
          a0 = a1 = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
          a0[i] = fmaf(v, w0[u][i], a0[i]);
          a1[i] = fmaf(v, w1[u][i], a1[i]);
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) pr[u] = nx[u];
    }
    put();
  }
};

// The shares that start inside a column with the tile's entries [a0, a1): k0 .. k1 - 1.
__device__ inline void fu_cut_by(int a0, int a1, int share, float inv, int& k0, int& k1) {
  auto quot = [&](int x) {  // x / share (the float quotient is off by one at most)
    int q = (int)((float)x * inv);
    if (q * share > x) q--;
    if ((q + 1) * share <= x) q++;
    return q;
  };
  k0 = quot(a0) + 1;
  k1 = quot(a1 - 1) + 1;
}

// Block pairs of X^T X at 5 to 8 blocks, dealt to four waves: block rows W and 7 - W (where there is one) of
// the upper triangle.  The most a wave has.
__host__ __device__ constexpr int fuw_pairs(int nb) { return nb == 8 ? 9 : nb == 7 ? 7 : nb == 6 ? 6 : 5; }
template <class F>
__device__ inline void fuw_for_wave(int wave, F&& f) {
  switch (wave) {
    case 0: f(std::integral_constant<int, 0>{}); break;
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    default: f(std::integral_constant<int, 3>{}); break;
  }
}

}  // namespace dn
