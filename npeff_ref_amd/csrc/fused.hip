// The factorisation step at ranks up to 128 (above 64: the updates of fused_wide.hip): three or four launches per iteration.
//
//   k_fu_n     A H^T as sums over chunks of a row's entries; its first workgroups sum the partial
//              Gram matrices of H that the last H update left
//   k_fu_w     W update: chunk sums, W G_H, the multiplicative update, and W^T W of the new W
//   k_fu_sum   sums the partial Gram matrices of W (only where there are more than a few)
//   k_fu_h     H update: A^T W of 64 columns gathered into LDS, H G_W, the update, and H^T H of the
//              new H; A^T W never goes through memory and H is read once and written once
//
// The separate kernels move five times the factor per H update (A^T W written and read, H read twice,
// written once) and need some ten launches per iteration, which is what bounds small problems.
//
// Matrix products run on the fp32 matrix cores (v_mfma_f32_16x16x4f32) with the factor's row as column
// operand: lane (j = l % 16, g = l / 16) holds components 16 b + 4 g + i of row j, which is both what
// the instruction wants as operand (with the contraction index permuted alike on both sides) and how
// it returns the product.  A rank that is not a multiple of 16 leaves rem components in the last
// block: they are dealt R = ceil(rem / 4) to a lane, so that the block takes R instead of four
// contraction steps.  Rows are read and written with 16-byte accesses whatever the rank (global memory
// needs no more than 4-byte alignment); the arrays end with four spare floats.
//
// All sums run in an order that the matrix and the launch shape fix: runs repeat bit for bit.
#include "fused.hpp"

#include <algorithm>
#include <cstdio>

namespace dn {

constexpr int FU_ROWS_WG = 64;       // rows of a workgroup of the W update
// Partial Gram matrices of W that the H update sums by itself (5 of them at 300 x 146k, r = 20: half a us where k_fu_sum
// takes 3.3; above two blocks every workgroup would read 80 KB).
constexpr int fu_sum_direct(int nb) { return nb > 2 ? 4 : 8; }

__host__ __device__ constexpr int fu_blocks(int Q, int R) { return Q + (R ? 1 : 0); }
// Lanes that cover a row of W with two 16-byte pieces each.
__host__ __device__ constexpr int fu_lpr(int Q, int R) {
  return 16 * Q + 4 * R <= 8 ? 1 : 16 * Q + 4 * R <= 16 ? 2 : 16 * Q + 4 * R <= 32 ? 4 : 8;
}

// G as the A operand of the products: [block b of output components][contraction block q][lane][i].
// part: n_parts partial matrices of packed upper block pairs ([pair][16][16]), summed in fp64 in order.
// They are read in 16-byte pieces, up to eight parts at a time, and come to their places through `stage` (as
// much LDS as a packed matrix, free again when this returns): with every thread picking its numbers from memory
// the vector-memory unit was busy for 16 lines per load (5 parts, 300 x 146k, r = 20: H update 23.6 us, now 20.0).
// All pieces of a thread are asked for together, and a single matrix once: piece after piece, four parts each, ten iterations at
// 500 x 2000, r = 64, took 355 us, now 337.
template <int Q, int R>
__device__ inline void fu_load_g(const float* __restrict__ part, int n_parts, int r, float* __restrict__ ga,
                                 float* __restrict__ stage) {
  constexpr int NB = fu_blocks(Q, R), S = fu_pairs(NB) * 256, N = NB * NB, P = NB > 2 ? 4 : 8;
  if constexpr (NB == 1) {  // (one number per thread: no detour)
    const int i = threadIdx.x & 3, rho = (threadIdx.x >> 2) & 15, g = threadIdx.x >> 6;
    const int k = R == 0 ? 4 * g + i : R * g + i, c = R == 0 ? rho : R * (rho >> 2) + (rho & 3);
    const bool ok = k < r && c < r && (R == 0 || (i < R && (rho & 3) < R));
    const float* src = part + (ok ? k * 16 + c : 0);
    double sum = 0.0;
    if (n_parts == 1) sum = (double)*src;
    else
      for (int p = 0; p < n_parts; p += P) {
        float v[P];
#pragma unroll
        for (int u = 0; u < P; u++) v[u] = src[(int64_t)(p + u < n_parts ? p + u : p) * S];
#pragma unroll
        for (int u = 0; u < P; u++) sum += p + u < n_parts ? (double)v[u] : 0.0;
      }
    ga[threadIdx.x] = ok ? (float)sum : 0.0f;
    return;
  }
  constexpr int PIECES = (S + 1023) / 1024;
  const int first = 4 * (int)threadIdx.x;
  auto at = [&](int j) { return first + 1024 * j < S ? first + 1024 * j : 0; };
  f32x4 g[PIECES];
  if (n_parts == 1) {
#pragma unroll
    for (int j = 0; j < PIECES; j++) g[j] = *reinterpret_cast<const f32x4*>(part + at(j));
  } else {
    double sum[PIECES][4] = {};
    for (int p = 0; p < n_parts; p += P) {
      f32x4 v[P][PIECES];
#pragma unroll
      for (int k = 0; k < P; k++)
#pragma unroll
        for (int j = 0; j < PIECES; j++) v[k][j] = *reinterpret_cast<const f32x4*>(part + (int64_t)(p + k < n_parts ? p + k : p) * S + at(j));
#pragma unroll
      for (int k = 0; k < P; k++)
#pragma unroll
        for (int j = 0; j < PIECES; j++)
#pragma unroll
          for (int i = 0; i < 4; i++) sum[j][i] += p + k < n_parts ? (double)v[k][j][i] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < PIECES; j++) g[j] = f32x4{(float)sum[j][0], (float)sum[j][1], (float)sum[j][2], (float)sum[j][3]};
  }
#pragma unroll
  for (int j = 0; j < PIECES; j++)
    if (first + 1024 * j < S) *reinterpret_cast<f32x4*>(stage + first + 1024 * j) = g[j];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < N; u++) {
    const int i = threadIdx.x & 3, lane = (threadIdx.x >> 2) & 63, q = u % NB, b = u / NB;
    const int rho = lane & 15, g = lane >> 4;
    int k, c;
    bool ok = true;
    if (R == 0 || q < Q) k = 16 * q + 4 * g + i;
    else { k = 16 * Q + R * g + i; ok = i < R; }
    if (R == 0 || b < Q) c = 16 * b + rho;
    else { c = 16 * Q + R * (rho >> 2) + (rho & 3); ok = ok && (rho & 3) < R; }
    ok = ok && k < r && c < r;
    const int bk = k >> 4, bc = c >> 4;
    const int x = bk <= bc ? fu_pair(bk, bc, NB) * 256 + (k & 15) * 16 + (c & 15)
                           : fu_pair(bc, bk, NB) * 256 + (c & 15) * 16 + (k & 15);
    ga[threadIdx.x + 256 * u] = ok ? stage[x] : 0.0f;
  }
  __syncthreads();
}

// The components of one factor row that a lane holds: x[b][i] = row[component(b, g, i)], zero past r.
template <int Q, int R>
__device__ inline void fu_load_row(const float* __restrict__ row, int g, int r, f32x4 (&x)[fu_blocks(Q, R)]) {
  constexpr int NB = fu_blocks(Q, R);
#pragma unroll
  for (int b = 0; b < Q; b++) {
    x[b] = *reinterpret_cast<const f32x4u*>(row + 16 * b + 4 * g);
    if (R == 0 && b == Q - 1) {
#pragma unroll
      for (int i = 0; i < 4; i++) x[b][i] = 16 * b + 4 * g + i < r ? x[b][i] : 0.0f;
    }
  }
  if constexpr (R > 0) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int c = 16 * Q + R * g + i;
      x[NB - 1][i] = i < R && c < r ? row[c] : 0.0f;
    }
  }
}

// PAST: the new rows go past the L2s, which write back what is left in them when the launch ends.  That pays while they
// hold the whole factor (32 MB together); of a larger one most is written back by then.  Ten iterations without / with: 342 /
// 330 us at 500 x 234k, r = 16 (14 MB), 391 / 377 at 300 x 175k, r = 20 (21 MB), 418 / 403 at 500 x 328k, r = 8 (20 MB), 435 /
// 428 at 300 x 399k, r = 8 (24 MB), 442 / 436 at 500 x 47k, r = 50 (11 MB); 497 / 505 at 300 x 402k, r = 16 (25 MB),
// 686 / 705 at 300 x 643k, r = 16 (39 MB), 968 / 997 at 500 x 1.0M, r = 16 (61 MB),
// 1721 / 1874 at 1500 x 1.1M, r = 32 (135 MB).
constexpr int64_t FU_PAST_BYTES = 24 << 20;
template <bool PAST>
__device__ inline void fu_store(float* dst, float v) {
  if constexpr (PAST) __builtin_nontemporal_store(v, dst);
  else *dst = v;
}
template <bool PAST>
__device__ inline void fu_store4(float* dst, const f32x4& v) {
  if constexpr (PAST) __builtin_nontemporal_store(f32x4u(v), reinterpret_cast<f32x4u*>(dst));
  else *reinterpret_cast<f32x4u*>(dst) = v;
}

// X G, the update and the new row for the 16 rows of a wave.  t: the numerators of the lane's row, laid
// out as x.  The new rows go to `dst` (global, if store) and into the wave's part of the LDS tile
// ([row][component], stride TS), from where they enter the Gram products.
template <int Q, int R, bool PAST = false>
__device__ inline void fu_update(const float* __restrict__ ga, f32x4 (&x)[fu_blocks(Q, R)],
                                 const f32x4 (&t)[fu_blocks(Q, R)], float eps, int r, bool store,
                                 float* __restrict__ dst, float* __restrict__ tile_row) {
  constexpr int NB = fu_blocks(Q, R);
  const int lane = threadIdx.x & 63, g = lane >> 4;
  f32x4 d[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) d[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int q = 0; q < NB; q++) {
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(ga + ((b * NB + q) * 64 + lane) * 4);
#pragma unroll
      for (int i = 0; i < (q < Q ? 4 : R); i++)
        d[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], x[q][i], d[b], 0, 0, 0);
    }
  }
#pragma unroll
  for (int b = 0; b < NB; b++) {
    f32x4 y;
    const f32x4 q = mu_quotients(t[b], d[b] + eps);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int c = b < Q ? 16 * b + 4 * g + i : 16 * Q + R * g + i;
      const float v = x[b][i] * q[i];
      const bool in = R > 0 ? b < Q || (i < R && c < r) : b < Q - 1 || c < r;
      y[i] = store && in ? v : 0.0f;
    }
    if (b < Q) {
      *reinterpret_cast<f32x4*>(tile_row + 16 * b + 4 * g) = y;
      if (store) {
        if (R > 0 || b < Q - 1 || 16 * b + 4 * g + 3 < r) fu_store4<PAST>(dst + 16 * b + 4 * g, y);
        else {
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (16 * b + 4 * g + i < r) fu_store<PAST>(dst + 16 * b + 4 * g + i, y[i]);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < R; i++) {
        const int c = 16 * Q + R * g + i;
        tile_row[c] = y[i];
        if (store && c < r) fu_store<PAST>(dst + c, y[i]);
      }
    }
  }
}

// acc += the Gram blocks of the 16 rows of the wave's part of the tile.
template <int NB>
__device__ inline void fu_gram(const float* __restrict__ rows, int ts, f32x4 (&acc)[fu_pairs(NB)]) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int s = 0; s < 4; s++) {
    float a[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) a[b] = rows[(4 * s + g) * ts + 16 * b + l16];
    int p = 0;
#pragma unroll
    for (int b1 = 0; b1 < NB; b1++)
#pragma unroll
      for (int b2 = b1; b2 < NB; b2++, p++)
        acc[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b1], a[b2], acc[p], 0, 0, 0);
  }
}

// sum += acc, acc = 0
template <int NP>
__device__ inline void fu_gram_fold(double (&sum)[NP][4], f32x4 (&acc)[NP]) {
#pragma unroll
  for (int p = 0; p < NP; p++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      sum[p][i] += (double)acc[p][i];
      acc[p][i] = 0.0f;
    }
}

// The four waves' Gram blocks, added in fp64 in wave order, to out ([pair][16][16]).  All waves' blocks through
// LDS at once where the tile's share of it holds them (fu_out_floats); else one wave after the other.
template <int NP, class T>
constexpr int fu_out_floats(int room) {
  return NP * 1024 * (int)(sizeof(T) / sizeof(float)) <= room ? NP * 1024 * (int)(sizeof(T) / sizeof(float)) : NP * 512;
}
template <int NP, int ROOM, class T, class V>
__device__ inline void fu_gram_out(const V& v, float* __restrict__ lds, float* __restrict__ out) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  if constexpr (fu_out_floats<NP, T>(ROOM) > NP * 512) {
    T* all = reinterpret_cast<T*>(lds);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; p++)
#pragma unroll
      for (int i = 0; i < 4; i++) all[(wave * NP + p) * 256 + (4 * g + i) * 16 + l16] = v[p][i];
    __syncthreads();
    for (int x = threadIdx.x; x < NP * 256; x += 256) {
      double s = (double)all[x];
#pragma unroll
      for (int w = 1; w < 4; w++) s += (double)all[w * NP * 256 + x];
      out[x] = (float)s;
    }
    return;
  }
  double* sum = reinterpret_cast<double*>(lds);
  for (int w = 0; w < 4; w++) {
    __syncthreads();
    if (wave == w) {
#pragma unroll
      for (int p = 0; p < NP; p++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          double* at = sum + p * 256 + (4 * g + i) * 16 + l16;
          *at = w == 0 ? (double)v[p][i] : *at + (double)v[p][i];
        }
    }
  }
  __syncthreads();
  for (int x = threadIdx.x; x < NP * 256; x += 256) out[x] = (float)sum[x];
}

// ---------------------------------------------------------------------------
// H update.  A tile is up to TC = 64 JB columns that share one aligned group of TC, with up to 16 TC
// entries (or one longer column); every wave has 16 JB of the group's columns.  The tile's entries,
// column by column, are cut into equal shares for the lane groups of LPR lanes (16 bytes of a row of W
// per lane); a group adds the entries of a column up in registers and stores the sum to the tile when
// the column ends.  Columns hold 1 to n entries with a few on average, so whole columns per group would
// leave most groups waiting for the longest one (a group walked up to 256 entries by itself: 110 us
// at 300 rows); a column cut by a share's end leaves its later parts in `carry`, one per group, and
// whoever reads the column adds them in order.  U gathers per group are in flight, the pairs of the
// next U are requested behind them, and a tile's first pairs and offsets while the products of the
// tile before run: without that a tile is a chain of five dependent trips to memory.
//
// Bound by vector and matrix instructions (at r = 50 they hold the SIMDs for 32 and 37 % of the time), not by
// memory: hence 32 bytes per lane and gathered row (the index arithmetic and the test for the column's
// end are shared by eight components; with 16 bytes the r = 50 step took 335 us, now 316), 24-bit
// multiplies into 32-bit offsets and the corrected reciprocal in place of the division sequence
// (390 -> 335 us with it).  777 x 862k, r = 50: 188 us for 2.0 GFLOP of gathers and 12.9 of products
// (922 us for A^T W, update and Gram as separate kernels); 512 x 431k, r = 16: 32 us (139); 300 x 146k,
// r = 20: 18.4, of which a workgroup has 12 us (prologue 2.8, rows and gathers 4 to 8, products and stores 3.5).
//
// Which shares left a carry for a column (fu_cut_by) one thread per column finds before the entries are gathered, not every
// lane that updates a part of it: two quotients a lane were up to a tenth of the vector instructions (ten iterations at
// 512 x 431k, r = 16: 561 -> 554 us, 777 x 862k, r = 50: 2801 -> 2781, a job at 300 x 146k, r = 20: 4.26 -> 4.19 ms.  At
// ranks above 64 the kernel has no two registers for it: 27.4 -> 27.6 ms at 1000 x 3.4M, r = 128).
// ---------------------------------------------------------------------------
template <int Q, int R, int JB, bool TOTALS, bool PAST>
__global__ void __launch_bounds__(256, fu_blocks(Q, R) <= 2 ? 4 : 3)
    k_fu_h(const fu_tile* __restrict__ tiles, int n_tiles, const int64_t* __restrict__ colptr,
           const uint2* __restrict__ pairs, int r, const float* __restrict__ W, float* __restrict__ H, float eps,
           const float* __restrict__ gw, int n_gw, float* __restrict__ gpart) {
  constexpr int NB = fu_blocks(Q, R), NP = fu_pairs(NB), TS = 16 * NB + 4, TC = 64 * JB;
  using Gather = fu_gather<TC, TS, NB, fu_lpr(Q, R)>;
  using Out = std::conditional_t<TOTALS, double, float>;
  constexpr int ROOM = Gather::CARRY + 2048, T_OUT = fu_out_floats<NP, Out>(ROOM), T_FLOATS = ROOM > T_OUT ? ROOM : T_OUT;
  __shared__ __align__(16) float ga[NB * NB * 256];
  __shared__ __align__(16) float tile[T_FLOATS];
  // Of the tile's columns: the first share that left a carry and, above 16 bits, the one past the last; -1 without entries.
  __shared__ int cut[2][TC];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, g = lane >> 4;
  double sum[TOTALS ? NP : 1][4] = {};
  f32x4 acc[NP];
#pragma unroll
  for (int p = 0; p < NP; p++) acc[p] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const char* Wb = reinterpret_cast<const char*>(W);
  Gather gather;
  gather.init(r);
  static_assert(TC <= 256, "a thread per column");
  int64_t cp0, cp1;  // entries of column tid of the tile
  auto request = [&](const fu_tile_at& d) {
    gather.request(pairs, d);
    const int64_t* at = colptr + d.col0 + (tid < d.nc ? tid : 0);
    cp0 = at[0];
    cp1 = at[1];
  };
  fu_tile_at td = fu_describe<Gather::NG>(tiles, n_tiles, blockIdx.x);
  request(td);
  fu_load_g<Q, R>(gw, n_gw, r, ga, tile);

  int par = 0;
  for (int tl = blockIdx.x; tl < n_tiles; tl += gridDim.x, par ^= 1) {
    const int l0 = td.col0 & (TC - 1);
    const int nc = td.nc;
    if (tid < nc) {
      const int a0 = (int)(cp0 - td.e0), a1 = (int)(cp1 - td.e0);
      int k0 = 0, k1 = -1;
      if (a1 > a0) fu_cut_by(a0, a1, td.share, 1.0f / (float)td.share, k0, k1);
      cut[par][l0 + tid] = k0 | (int)((unsigned)k1 << 16);
    }
    const fu_tile_at nd = fu_describe<Gather::NG>(tiles, n_tiles, tl + gridDim.x);
    // the wave's rows of H
    const int64_t base = td.col0 - l0;
    float* Hb = H + base * r;
    f32x4 h[JB][NB];
    bool mine[JB];
    unsigned hoff[JB];
#pragma unroll
    for (int jb = 0; jb < JB; jb++) {
      const int jl = 16 * (JB * wave + jb) + l16;
      mine[jb] = jl >= l0 && jl < l0 + nc;
      hoff[jb] = (unsigned)(mine[jb] ? jl : l0) * (unsigned)r;
      fu_load_row<Q, R>(Hb + hoff[jb], g, r, h[jb]);
    }

    gather.template run<0>(pairs, td, Wb, tile);
    request(nd);
    __syncthreads();

#pragma unroll
    for (int jb = 0; jb < JB; jb++) {
      const int first = 16 * (JB * wave + jb);
      if (first + 15 < l0 || first >= l0 + nc) continue;
      f32x4 t[NB];
      float* trow = tile + (first + l16) * TS;
      const int parts = mine[jb] ? cut[par][first + l16] : -1;
      const bool some = parts >= 0;
#pragma unroll
      for (int b = 0; b < Q; b++) t[b] = *reinterpret_cast<const f32x4*>(trow + 16 * b + 4 * g);
      if constexpr (R > 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) t[NB - 1][i] = i < R ? trow[16 * Q + R * g + i] : 0.0f;
      }
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int i = 0; i < 4; i++) t[b][i] = some ? t[b][i] : 0.0f;
      if (some) {
        const int k0 = parts & 0xffff, k1 = parts >> 16;
        auto add = [&](int k, f32x4 (&to)[NB]) {
          const float* src = tile + Gather::CARRY + k * (2048 / Gather::NG);
#pragma unroll
          for (int b = 0; b < NB; b++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
              if (b < Q || i < R) to[b][i] += src[b < Q ? 16 * b + 4 * g + i : 16 * Q + R * g + i];
            }
        };
        if (NB > 2 || !__any(k1 - k0 > 16)) {
          for (int k = k0; k < k1; k++) add(k, t);
        } else {
          // The parts of a long column eight at a time: one by one the sum rounds as often as it has parts
          // (62 for 2000 rows at r = 16, where the update was off by 1.3e-7, now 9.8e-8).
          for (int k = k0; k < k1;) {
            f32x4 part[NB];
#pragma unroll
            for (int b = 0; b < NB; b++) part[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            for (const int k8 = k + 8; k < k1 && k < k8; k++) add(k, part);
#pragma unroll
            for (int b = 0; b < NB; b++) t[b] += part[b];
          }
        }
      }
      fu_update<Q, R, PAST>(ga, h[jb], t, eps, r, mine[jb], Hb + hoff[jb], trow);
      __builtin_amdgcn_wave_barrier();
      fu_gram<NB>(tile + first * TS, TS, acc);
    }
    if constexpr (TOTALS) fu_gram_fold<NP>(sum, acc);
    td = nd;
    __syncthreads();  // (the tile has been read)
  }
  float* out = gpart + (int64_t)blockIdx.x * (NP * 256);
  if constexpr (TOTALS) fu_gram_out<NP, ROOM, double>(sum, tile, out);
  else fu_gram_out<NP, ROOM, float>(acc, tile, out);
}

// W update: 64 rows per workgroup.  n_base (or NULL: N holds A H^T itself): first chunk of every row.
template <int Q, int R>
__global__ void __launch_bounds__(256)
    k_fu_w(int64_t n, int r, const int* __restrict__ n_base, const float* __restrict__ N, float* __restrict__ W,
           float eps, const float* __restrict__ gh, int n_gh, float* __restrict__ gpart) {
  constexpr int NB = fu_blocks(Q, R), NP = fu_pairs(NB), TS = 16 * NB + 4;
  constexpr int T_OUT = NP * 1024, T_FLOATS = FU_ROWS_WG * TS > T_OUT ? FU_ROWS_WG * TS : T_OUT;
  __shared__ __align__(16) float ga[NB * NB * 256];
  __shared__ __align__(16) float tile[T_FLOATS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * FU_ROWS_WG;
  const int64_t i = row0 + 16 * wave + l16;
  const bool mine = i < n;
  const int64_t at = mine ? i : row0;
  const int k0 = n_base ? n_base[at] : (int)at, k1 = n_base ? n_base[at + 1] : (int)at + 1;
  f32x4 x[NB], t[NB];
  float* wrow = W + at * r;
  fu_load_row<Q, R>(wrow, g, r, x);
  fu_load_g<Q, R>(gh, n_gh, r, ga, tile);
#pragma unroll
  for (int b = 0; b < NB; b++) t[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int U = 4;  // chunk sums asked for at a time (one by one they are a chain of trips to memory)
  for (int k = k0; k < k1; k += U) {
    f32x4 p[U][NB];
#pragma unroll
    for (int u = 0; u < U; u++) fu_load_row<Q, R>(N + (int64_t)(k + u < k1 ? k + u : k) * r, g, r, p[u]);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int c = 0; c < 4; c++) t[b][c] += k + u < k1 ? p[u][b][c] : 0.0f;
  }
  f32x4 acc[NP];
#pragma unroll
  for (int p = 0; p < NP; p++) acc[p] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  __syncthreads();
  fu_update<Q, R>(ga, x, t, eps, r, mine, wrow, tile + (16 * wave + l16) * TS);
  __builtin_amdgcn_wave_barrier();
  fu_gram<NB>(tile + 16 * wave * TS, TS, acc);
  fu_gram_out<NP, T_OUT, float>(acc, tile, gpart + (int64_t)blockIdx.x * (NP * 256));
}

// Element x of the sum of n_parts partial Gram matrices: 16 elements per workgroup, 16 threads each.
__device__ inline void fu_sum_parts(const float* __restrict__ part, int n_parts, int S, int block,
                                    float* __restrict__ out, double* __restrict__ red) {
  const int x = block * 16 + (threadIdx.x & 15), k = threadIdx.x >> 4;
  const float* p = part + x;
  double s = 0.0;
  for (int q = k; q < n_parts; q += 16 * 16) {  // (sixteen parts at a time under way)
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) v[u] = p[(int64_t)(q + 16 * u < n_parts ? q + 16 * u : q) * S];
#pragma unroll
    for (int u = 0; u < 16; u++) s += q + 16 * u < n_parts ? (double)v[u] : 0.0;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < 16) {
    for (int u = 1; u < 16; u++) s += red[16 * u + threadIdx.x];
    out[x] = (float)s;
  }
}

__global__ void __launch_bounds__(256)
    k_fu_sum(const float* __restrict__ part, int n_parts, int S, float* __restrict__ out) {
  __shared__ double red[256];
  fu_sum_parts(part, n_parts, S, blockIdx.x, out, red);
}

// X^T X of a factor that no update of the step has left, `per` rows (a multiple of 64) per workgroup, as
// partial matrices like the updates'.  The fp32 sums of 256 rows are added up in fp64.
//
// Up to 4 blocks of 16 components each wave takes every fourth 16 rows and all block pairs; the operands
// need no LDS there: a lane's number of a row is one 4-byte load, 16 lanes a whole sector.  861,696 x 50 in
// 80 us (708 with k_gram), 429,626 x 16 in 9 (36).
template <int NB>
__global__ void __launch_bounds__(256)
    k_fu_gram(const float* __restrict__ X, int64_t rows, int64_t per, int r, float* __restrict__ gpart) {
  constexpr int NP = fu_pairs(NB);
  __shared__ __align__(16) float lds[NP * 512];
  const int64_t row0 = blockIdx.x * per, row1 = row0 + per < rows ? row0 + per : rows;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  float a[4][NB], nx[4][NB];
  auto load = [&](int64_t base, float (&v)[4][NB]) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int64_t row = base + 4 * s + g;
#pragma unroll
      for (int b = 0; b < NB; b++)
        v[s][b] = X[row < row1 && 16 * b + l16 < r ? row * r + 16 * b + l16 : 0];
    }
  };
  double sum[NP][4] = {};
  f32x4 acc[NP] = {};
  int64_t base = row0 + 16 * (int)(threadIdx.x >> 6);
  load(base, a);
  for (int k = 1; base < row1; base += 64, k++) {
    load(base + 64, nx);
#pragma unroll
    for (int s = 0; s < 4; s++) {
#pragma unroll
      for (int b = 0; b < NB; b++) a[s][b] = base + 4 * s + g < row1 && 16 * b + l16 < r ? a[s][b] : 0.0f;
      int p = 0;
#pragma unroll
      for (int b1 = 0; b1 < NB; b1++)
#pragma unroll
        for (int b2 = b1; b2 < NB; b2++, p++)
          acc[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][b1], a[s][b2], acc[p], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < NB; b++) a[s][b] = nx[s][b];
    }
    if (k % 16 == 0) fu_gram_fold<NP>(sum, acc);
  }
  fu_gram_fold<NP>(sum, acc);
  fu_gram_out<NP, 0, double>(sum, lds, gpart + (int64_t)blockIdx.x * (NP * 256));
}

// 5 to 8 blocks: all waves take the same rows, 32 at a time through LDS (rows 16 banks apart: the four
// rows of an operand do not meet), and their share of the pairs, block rows W and 7 - W.  Bound by the fp32
// matrix cores (400 us of them at 3.4 M x 128): 597 us (1362 with k_gram; 964 with every wave's operands
// straight from global memory, one trip of latency for 36 matrix instructions).
constexpr int FU_GRAM_ROWS = 32;
constexpr int fu_gram_stride(int nb) { return 16 * (nb | 1); }

template <int NB>
__global__ void __launch_bounds__(256, 2)
    k_fu_gram_wide(const float* __restrict__ X, int64_t rows, int64_t per, int r, float* __restrict__ gpart) {
  constexpr int NA = fuw_pairs(NB), LD = fu_gram_stride(NB);
  __shared__ __align__(16) float lds[2 * FU_GRAM_ROWS * LD];
  const int64_t row0 = blockIdx.x * per, row1 = row0 + per < rows ? row0 + per : rows;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int c4 = 4 * (tid & 31), lr = tid >> 5;  // loader: four components of every eighth row
  f32x4 st[4];
  auto fetch = [&](int64_t base) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int64_t row = base + lr + 8 * q;
      // (a row's last piece may end past it: the arrays have four spare floats)
      st[q] = *reinterpret_cast<const f32x4u*>(X + (row < row1 && c4 < r ? row * r + c4 : 0));
    }
  };
  auto commit = [&](int64_t base, float* to) {  // (zeros past the rows and the rank put in here: the loads stay on their way)
    if (c4 < 16 * NB) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = base + lr + 8 * q < row1 && c4 + i < r ? st[q][i] : 0.0f;
        *reinterpret_cast<f32x4*>(to + (lr + 8 * q) * LD + c4) = v;
      }
    }
  };
  double sum[NA][4] = {};
  f32x4 acc[NA] = {};
  fetch(row0);
  commit(row0, lds);
  fetch(row0 + FU_GRAM_ROWS);
  __syncthreads();
  int k = 0;
  for (int64_t base = row0; base < row1; base += FU_GRAM_ROWS, k++) {
    const float* at = lds + (k & 1) * FU_GRAM_ROWS * LD + g * LD + l16;
    fuw_for_wave(wave, [&](auto w) {
      constexpr int W = decltype(w)::value, W1 = 7 - W;
      float a[2][NB];  // the next rows' operands are read ahead of the matrix instructions
      auto read = [&](int s, float (&v)[NB]) {
#pragma unroll
        for (int b = W; b < NB; b++) v[b] = at[4 * s * LD + 16 * b];
      };
      read(0, a[0]);
#pragma unroll
      for (int s = 0; s < FU_GRAM_ROWS / 4; s++) {
        const float (&v)[NB] = a[s & 1];
        if (s + 1 < FU_GRAM_ROWS / 4) read(s + 1, a[(s + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = W; b < NB; b++) {
          acc[b - W] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[W], v[b], acc[b - W], 0, 0, 0);
          if constexpr (W1 < NB) {
            if (b >= W1) acc[NB - W + b - W1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[W1], v[b], acc[NB - W + b - W1], 0, 0, 0);
          }
        }
      }
    });
    // (the other buffer was last read before the barrier that ended the step before)
    commit(base + FU_GRAM_ROWS, lds + ((k + 1) & 1) * FU_GRAM_ROWS * LD);
    fetch(base + 2 * FU_GRAM_ROWS);
    if (k % 8 == 7) fu_gram_fold<NA>(sum, acc);
    __syncthreads();
  }
  fu_gram_fold<NA>(sum, acc);
  float* out = gpart + (int64_t)blockIdx.x * (fu_pairs(NB) * 256);
  auto put = [&](int b1, int b2, const double (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) out[fu_pair(b1, b2, NB) * 256 + (4 * g + i) * 16 + l16] = (float)v[i];
  };
  fuw_for_wave(wave, [&](auto w) {
    constexpr int W = decltype(w)::value, W1 = 7 - W;
#pragma unroll
    for (int b = W; b < NB; b++) put(W, b, sum[b - W]);
    if constexpr (W1 < NB) {
#pragma unroll
      for (int b = W1; b < NB; b++) put(W1, b, sum[NB - W + b - W1]);
    }
  });
}

// A H^T: chunk blockIdx.x - sum_wgs of the entries, all of one row (XCD: a part of a row's share of an XCD's
// columns); the wave's lane groups take them round-robin, FU_U gathers each in flight.  Workgroups 0 .. sum_wgs - 1 sum
// Gram parts instead.  777 x 862k, r = 50, in chunks of whole rows: 117 us for 3.9 M gathered rows of 200 bytes (6.6 TB/s),
// half of which the L2s hold; 141 us as one 4-byte load per lane; by XCD 75.
template <int LPR, bool XCD>
__global__ void __launch_bounds__(256)
    k_fu_n(const fu_chunk* __restrict__ chunks, const int64_t* __restrict__ x_seg, int x_parts,
           const int32_t* __restrict__ colind, const float* __restrict__ vals, int r, const float* __restrict__ H,
           float* __restrict__ N, int sum_wgs, const float* __restrict__ part, int n_parts, int S,
           float* __restrict__ gsum) {
  __shared__ __align__(16) double red_d[256];
  if ((int)blockIdx.x < sum_wgs) {
    if ((int)blockIdx.x < S / 16) fu_sum_parts(part, n_parts, S, blockIdx.x, gsum, red_d);
    return;
  }
  constexpr int G = 64 / LPR;
  // A lane group adds up 64 entries at a time and their sums in LDS: one sum over its share of a chunk, 1000
  // entries of 32 M at r = 90, left the W update at 2000 x 0.5 M with an error of 1.0e-6 (now 2.5e-7; 117.4
  // against 115.6 us at the size above).
  __shared__ __align__(16) float totals[256][4];
  float* red = reinterpret_cast<float*>(red_d);  // [4][4 LPR]
  int64_t chunk = blockIdx.x - sum_wgs, e0;
  int len;
  if constexpr (XCD) {  // (sum_wgs is a multiple of 8)
    const unsigned u = (unsigned)chunk >> 3, x = (unsigned)chunk & 7, row = u / (unsigned)x_parts, k = u % (unsigned)x_parts;
    const int64_t s0 = x_seg[8 * row + x], s1 = x_seg[8 * row + x + 1], each = (unsigned)(s1 - s0 + x_parts - 1) / (unsigned)x_parts;
    e0 = s0 + k * each;
    len = (int)(e0 >= s1 ? 0 : e0 + each < s1 ? each : s1 - e0);
    chunk = (8 * row + x) * (unsigned)x_parts + k;
  } else {
    e0 = chunks[chunk].e0;
    len = chunks[chunk].len;
  }
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, sub = lane % LPR, grp = lane / LPR;
  const float* Hl = H + (4 * sub < r ? 4 * sub : 0);  // (lanes past the rank: any valid address)
  const int per = (len + 3) / 4;
  const int w0 = wave * per, w1 = w0 + per < len ? w0 + per : len;
  const int32_t* ci = colind + e0;
  const float* va = vals + e0;
  f32x4 a = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // 64 (column, value) pairs at a time, one per lane, the next 64 on their way; the steps take theirs by
  // shuffles.  Lanes past the end hold some column and are not counted in.
  if (w0 < w1) {
    auto request = [&](int e, int& jj, float& vv) {
      const int at = e + lane < w1 ? e + lane : w1 - 1;
      jj = ci[at];
      vv = va[at];
    };
    int j, jn;
    float v, vn;
    request(w0, j, v);
    int run = G;
    bool more = false;
    for (int b = w0; b < w1; b += 64) {
      if (run-- == 0) {
        f32x4* t = reinterpret_cast<f32x4*>(totals[tid]);
        *t = more ? *t + a : a;
        a = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        more = true;
        run = G - 1;
      }
      request(b + 64, jn, vn);
      const int cnt = w1 - b < 64 ? w1 - b : 64, steps = (cnt + G - 1) / G;
      constexpr int U = 64 / G < FU_U ? 64 / G : FU_U;
      for (int st = 0; st < steps; st += U) {
        f32x4 x[U];
        float w[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int src = ((st + u) * G + grp) & 63;
          const int64_t row = __shfl(j, src);
          w[u] = __shfl(v, src);
          x[u] = *reinterpret_cast<const f32x4u*>(Hl + row * r);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          if ((st + u) * G + grp >= cnt) continue;  // (0 times an infinite entry is no 0)
#pragma unroll
          for (int i = 0; i < 4; i++) a[i] = fmaf(w[u], x[u][i], a[i]);
        }
      }
      j = jn;
      v = vn;
    }
    if (more) a += *reinterpret_cast<f32x4*>(totals[tid]);
  }
#pragma unroll
  for (int off = 32; off >= LPR; off >>= 1)
#pragma unroll
    for (int i = 0; i < 4; i++) a[i] += __shfl_xor(a[i], off);
  if (grp == 0) *reinterpret_cast<f32x4*>(red + wave * 4 * LPR + 4 * sub) = a;
  __syncthreads();
  if (tid < r) N[chunk * r + tid] = ((red[tid] + red[4 * LPR + tid]) + red[8 * LPR + tid]) + red[12 * LPR + tid];
}

// Loss: <A H^T, W> over the chunk sums (one partial per workgroup, 64 rows), then with <W^T W, H^T H>.
__global__ void __launch_bounds__(256)
    k_fu_dot(int64_t n, int r, const int* __restrict__ n_base, const float* __restrict__ N,
             const float* __restrict__ W, double* __restrict__ out) {
  __shared__ double red[256];
  const int64_t row0 = (int64_t)blockIdx.x * 16, rows = n - row0 < 16 ? n - row0 : 16;
  double s = 0.0;
  for (int x = threadIdx.x; x < rows * r; x += 256) {
    const int64_t i = row0 + x / r;
    const int c = x % r;
    const int64_t k0 = n_base ? n_base[i] : i, k1 = n_base ? n_base[i + 1] : i + 1;
    float t = 0.0f;
    for (int64_t k = k0; k < k1; k++) t += N[k * r + c];
    s += (double)t * (double)W[i * r + c];
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256)
    k_fu_loss(const double* __restrict__ part, int n_parts, int r, const float* __restrict__ gw,
              const float* __restrict__ gh, double* __restrict__ out2) {
  __shared__ double red[2][256];
  double neg = 0.0, pos = 0.0;
  for (int k = threadIdx.x; k < n_parts; k += 256) neg += part[k];
  int p = 0;
  const int nb = (r + 15) / 16;
  for (int b1 = 0; b1 < nb; b1++)
    for (int b2 = b1; b2 < nb; b2++, p++) {
      const int x = p * 256 + threadIdx.x;
      const int a = 16 * b1 + (threadIdx.x >> 4), b = 16 * b2 + (threadIdx.x & 15);
      if (a >= r || b >= r) continue;  // (not defined there)
      const double v = (double)gw[x] * (double)gh[x];
      pos += b1 == b2 ? v : 2.0 * v;
    }
  red[0][threadIdx.x] = neg;
  red[1][threadIdx.x] = pos;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      red[0][threadIdx.x] += red[0][threadIdx.x + o];
      red[1][threadIdx.x] += red[1][threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x < 2) out2[threadIdx.x] = red[threadIdx.x][0];
}

// ---------------------------------------------------------------------------
// Plan: tiles and packed entries of A^T W, chunks of A H^T
// ---------------------------------------------------------------------------
// Tiles of the aligned group of `tc` columns `grp`: f(first column, columns) for each, in order.  A tile ends before the
// column that would take it past `most` entries; a column longer than `alone` shares its tile with no other.  A wave per
// group, a lane for every 64th column: the end of a tile is the first of the columns that a ballot shows to be past it.
// (A thread per group, column after column: counting and making the tiles of 145 k columns took 19 and 30 us, now 10 and 11.)
template <class F>
__device__ inline void fu_split_group(const int64_t* __restrict__ colptr, int64_t m, int tc, int64_t most, int64_t alone,
                                      int64_t grp, F&& f) {
  constexpr int Q = 4;  // (tc <= 256)
  const int lane = threadIdx.x & 63;
  const int64_t j0 = grp * tc;
  const int n = (int)(j0 + tc < m ? tc : m - j0);
  int64_t end[Q], e0 = colptr[j0];
  uint64_t there[Q], apart[Q], lone_before = 0;  // columns of the group, and those that start a tile because of `alone`
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const bool in = 64 * q + lane < n;
    const int64_t* at = colptr + j0 + (in ? 64 * q + lane : 0);
    end[q] = at[1];
    there[q] = __ballot(in);
    const uint64_t lone = __ballot(in && at[1] - at[0] > alone);
    apart[q] = lone | lone << 1 | lone_before >> 63;
    lone_before = lone;
  }
  for (int s = 0;;) {
    int t = n;
#pragma unroll
    for (int q = Q - 1; q >= 0; q--) {
      uint64_t mask = (__ballot(end[q] - e0 > most) | apart[q]) & there[q];
      if (s >= 64 * q) mask = s - 64 * q >= 63 ? 0 : mask & (~0ull << (s - 64 * q + 1));
      if (mask) t = 64 * q + __builtin_ctzll(mask);
    }
    f(j0 + s, t - s, e0);
    if (t == n) break;
#pragma unroll
    for (int q = 0; q < Q; q++)
      if ((t - 1) >> 6 == q) e0 = __shfl(end[q], (t - 1) & 63);
    s = t;
  }
}

__global__ void __launch_bounds__(256)
    k_fu_count_tiles(const int64_t* __restrict__ colptr, int64_t m, int tc, int64_t most, int64_t alone, int64_t groups,
                     int* __restrict__ count) {
  for (int64_t grp = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); grp < groups; grp += 4 * (int64_t)gridDim.x) {
    int k = 0;
    fu_split_group(colptr, m, tc, most, alone, grp, [&](int64_t, int, int64_t) { k++; });
    if ((threadIdx.x & 63) == 0) count[grp] = k;
  }
}

__global__ void __launch_bounds__(256)
    k_fu_make_tiles(const int64_t* __restrict__ colptr, int64_t m, int tc, int64_t most, int64_t alone, int64_t groups,
                    const int64_t* __restrict__ first, fu_tile* __restrict__ tiles) {
  const bool writes = (threadIdx.x & 63) == 0;
  for (int64_t grp = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); grp < groups; grp += 4 * (int64_t)gridDim.x) {
    int64_t k = first[grp];
    fu_split_group(colptr, m, tc, most, alone, grp, [&](int64_t col, int cols, int64_t e0) {
      if (writes) {
        tiles[k].e0 = e0;
        tiles[k].col0 = (int32_t)col;
        tiles[k].cols = cols;
      }
      k++;
    });
    if (writes && grp == groups - 1) {
      tiles[k].e0 = colptr[m];
      tiles[k].col0 = (int32_t)m;
      tiles[k].cols = 0;
    }
  }
}

// 256 columns per row of workgroups: the column of an entry from the offsets of its group.  (Several
// workgroups where there are few groups: the group of the longest columns alone took 210 us of a job on a
// matrix of 0.6 M entries.)
__global__ void __launch_bounds__(256)
    k_fu_pack_entries(const int64_t* __restrict__ colptr, const int32_t* __restrict__ rowind,
                      const float* __restrict__ tvals, int64_t m, int64_t groups, uint2* __restrict__ pairs) {
  __shared__ int64_t cp[FU_GROUP + 1];
  for (int64_t grp = blockIdx.x; grp < groups; grp += gridDim.x) {
    const int64_t j0 = grp * FU_GROUP;
    __syncthreads();
    cp[threadIdx.x] = colptr[j0 + threadIdx.x < m ? j0 + threadIdx.x : m];
    if (threadIdx.x == 0) cp[FU_GROUP] = colptr[j0 + FU_GROUP < m ? j0 + FU_GROUP : m];
    __syncthreads();
    const int64_t e1 = cp[FU_GROUP];
    for (int64_t e = cp[0] + 256 * blockIdx.y + threadIdx.x; e < e1; e += 256 * gridDim.y) {
      int lo = 0, hi = FU_GROUP;  // last column that starts at or before e
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cp[mid] <= e) lo = mid; else hi = mid;
      }
      pairs[e] = make_uint2((unsigned)rowind[e] | ((unsigned)lo << FU_ROW_BITS), __float_as_uint(tvals[e]));
    }
  }
}

__global__ void __launch_bounds__(256)
    k_fu_make_chunks(const int64_t* __restrict__ rowptr, int64_t n, int64_t chunk, const int64_t* __restrict__ base,
                     fu_chunk* __restrict__ chunks, int* __restrict__ base32) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i > n) return;
  base32[i] = (int)base[i];
  if (i == n) return;
  int64_t e = rowptr[i];
  const int64_t e1 = rowptr[i + 1];
  for (int64_t k = base[i]; k < base[i + 1]; k++, e += chunk) {
    chunks[k].e0 = e;
    chunks[k].len = (int32_t)(e1 - e < chunk ? e1 - e : chunk);
  }
}

void fused_drop(dnpeff_csr* S) {
  fused_plan& f = S->fused;
  dfree(f.tiles); dfree(f.pairs); dfree(f.chunks); dfree(f.n_base);
  dfree(f.x_col); dfree(f.x_val); dfree(f.x_seg); dfree(f.x_base);
  f = fused_plan();
}

// Columns per tile: 256, 128 or 64 by the rank (a tile of the factor of about 16 KB; fewer columns
// would leave a workgroup with more trips to memory than work), 64 where larger tiles would leave
// compute units without one.
static int fu_tile_cols(int64_t m, int r) {
  const int tc = r <= 16 ? 256 : r <= 32 ? 128 : r <= 64 ? 64 : FUW_COLS;
  return m >= (int64_t)tc * 2 * n_cus() || tc < 64 ? tc : 64;
}

static int fused_tiles_make(dnpeff_csr* S, int tc, int64_t most, int64_t alone, bool with_first) {
  fused_plan& f = S->fused;
  hipStream_t st = stream();
  DN_CHECK(S->colptr && S->n_cols > 0, "matrix has no transposed copy");
  if (!f.tiles || f.tile_cols != tc || f.tile_most != most || f.tile_alone != alone || (with_first && f.h_first.empty())) {
    const int64_t m = S->n_cols, groups = ceil_div(m, tc);
    dbuf<int> count;
    dbuf<int64_t> first;
    DN_TRY(count.alloc(groups));
    DN_TRY(first.alloc(groups + 1));
    DN_CHECK(tc <= 256, "tiles of %d columns", tc);
    const dim3 grid((unsigned)std::min<int64_t>(ceil_div(groups, 4), 1 << 20)), block(256);
    hipLaunchKernelGGL(k_fu_count_tiles, grid, block, 0, st, S->colptr, m, tc, most, alone, groups, count.p);
    DN_LAUNCH_CHECK();
    unsigned long long* host = nullptr;
    DN_TRY(host_words(&host));
    int64_t* total = reinterpret_cast<int64_t*>(host);
    DN_TRY(scan_counts_i64(count, groups, first, total));
    f.h_first.clear();
    if (with_first) {
      f.h_first.resize((size_t)groups + 1);
      DN_HIP(copy_down(f.h_first.data(), first, sizeof(int64_t) * f.h_first.size()));
    }
    DN_HIP(hipStreamSynchronize(st));
    const int64_t n_tiles = *total;
    dfree(f.tiles);
    f.tiles = nullptr;
    DN_TRY(dmalloc(&f.tiles, n_tiles + 1));
    f.n_tiles = n_tiles;
    f.tile_cols = tc;
    f.tile_most = most;
    f.tile_alone = alone;
    hipLaunchKernelGGL(k_fu_make_tiles, grid, block, 0, st, S->colptr, m, tc, most, alone, groups, first.p, f.tiles);
    DN_LAUNCH_CHECK();
  }
  return 0;
}

int fused_tiles_build(dnpeff_csr* S, int r) {
  const int tc = fu_tile_cols(S->n_cols, r);
  // Entries per tile: 16 per column.  The 32 columns of a tile at ranks above 64 are the smallest
  // matrix operand: a denser matrix gets as many as leave every compute unit 16 tiles (2000 x 2M with 64 M
  // entries, r = 90: 57 against 63 ms; at r = 20 smaller tiles are the better ones, 16.4 against 18.6).
  int64_t most = 16 * tc;
  if (r > FUSED_NARROW_RANK && r <= FUSED_MAX_RANK) most = std::max<int64_t>(most, S->nnz / (16 * (int64_t)n_cus()));
  // Above rank 128 (A^T W alone, a wave per eighth of a tile's columns) as few as 64 where the tiles leave compute units without
  // work: ten iterations at 119 x 5.2k, rank 460, 2.40 -> 2.30 ms, 60 x 6k, rank 256, 1.62 -> 1.53.  Everywhere it costs
  // 1 to 2 % from 150 x 159k and 200 x 46k on.
  if (r > FUSED_MAX_RANK && S->n_cols < (int64_t)tc * 2 * n_cus())
    most = std::max<int64_t>(64, std::min<int64_t>(most, S->nnz / (8 * (int64_t)n_cus())));
  return fused_tiles_make(S, tc, most, r > FUSED_MAX_RANK ? SPMM_T_LONG : INT64_MAX, false);
}

int fused_tiles_first(dnpeff_csr* S) {
  return fused_tiles_make(S, S->fused.tile_cols, S->fused.tile_most, S->fused.tile_alone, true);
}

// Entries per workgroup of A H^T: about FU_CHUNKS workgroups in all, at least 256 entries each.
static int64_t fu_chunk_entries(int64_t nnz) { return std::max<int64_t>(256, ceil_div(ceil_div(nnz, FU_CHUNKS), 256) * 256); }

// A row's entries by the XCD that their columns belong to (16 columns each in turn), in their order, a workgroup per
// row: every wave takes a quarter, counts, and places its entries behind those of the waves before.
__device__ inline int fu_xcd_of(int col) { return (col >> 4) & 7; }
__global__ void __launch_bounds__(256)
    k_fu_xcd_split(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colind, const float* __restrict__ vals,
                   int64_t n, int parts, int32_t* __restrict__ x_col, float* __restrict__ x_val, int64_t* __restrict__ x_seg,
                   int* __restrict__ n_base) {
  __shared__ int count[4][8];
  const int64_t row = blockIdx.x, r0 = rowptr[row], r1 = rowptr[row + 1];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t per = (r1 - r0 + 3) / 4, e0 = r0 + wave * per < r1 ? r0 + wave * per : r1, e1 = e0 + per < r1 ? e0 + per : r1;
  int mine = 0;  // (lane x < 8: entries of XCD x)
  auto walk = [&](auto&& f) {
    for (int64_t e = e0; e < e1; e += 64) {
      const bool in = e + lane < e1;
      const int col = colind[in ? e + lane : e1 - 1], x = fu_xcd_of(col);
      const uint64_t here = __ballot(in), b0 = __ballot(x & 1), b1 = __ballot(x & 2), b2 = __ballot(x & 4);
      auto of = [&](int y) { return here & (y & 1 ? b0 : ~b0) & (y & 2 ? b1 : ~b1) & (y & 4 ? b2 : ~b2); };
      f(e, in, col, x, of);
    }
  };
  walk([&](int64_t, bool, int, int, auto of) { mine += __popcll(of(lane & 7)); });
  if (lane < 8) count[wave][lane] = mine;
  __syncthreads();
  int64_t at = r0;  // (lane x < 8: where the wave's next entry of XCD x goes)
  for (int y = 0; y < 8; y++)
    for (int w = 0; w < 4; w++) at += y < (lane & 7) || (y == (lane & 7) && w < wave) ? count[w][y] : 0;
  if (wave == 0 && lane < 8) {
    x_seg[8 * row + lane] = at;
    if (lane == 0) n_base[row] = (int)(8 * parts * row);
    if (row == n - 1 && lane == 0) {
      x_seg[8 * n] = r1;
      n_base[n] = (int)(8 * parts * n);
    }
  }
  walk([&](int64_t e, bool in, int col, int x, auto of) {
    const int64_t base = __shfl(at, x);
    if (in) {
      const int64_t to = base + __popcll(of(x) & ((1ull << lane) - 1ull));
      x_col[to] = col;
      x_val[to] = vals[e + lane];
    }
    at += __popcll(of(lane & 7));
  });
}

// A H^T by XCD: workgroups are dealt to the XCDs round-robin, and where each XCD has its own eighth of the
// columns its L2 fetches a row of H once for all that gather it (and from a part of H an eighth as large), where
// with chunks of whole rows every XCD fetches most of H.  The columns are dealt in sixteens: an eighth
// in one piece has all the rare columns on the last XCD, whose misses are then waited for (777 x 862k, r = 50: 126
// us; with columns dealt one by one two XCDs share every line of short rows).  k_fu_n at 777 x 862k, r = 50 / 512 x 431k, r = 16
// / 300 x 146k, r = 20: 74.7 / 17.2 / 10.2 us, in chunks of whole rows 117 / 21.5 / 11.0.
// Up to 96 components: above, runs amplify the rounding of every sum (20 iterations at 772 x 467k, r = 128, end 1.7e-5
// apart in the one order and the other, at r <= 64 5e-6 at most), and keep the order they have always had.
// Rows of FU_XCD_ROW entries or more on average, of which none is twice as long (a workgroup per row and XCD).  Ten iterations
// in chunks of whole rows / by XCD: 191 / 215 us at 200 rows of 200 entries, r = 8, 252 / 281 at 500 of 512, r = 16, 488 / 546 at
// 1000 of 1024, r = 32 (a workgroup has 128 entries then), 317 / 286 at 500 of 1800, r = 8, 896 / 811 at 2000 of 1800, r = 24,
// 1550 / 1357, r = 64, 796 / 754 at 300 of 2048, r = 64, 5880 / 5476 at 1000 of 4096, r = 96, 9751 / 8205 at 2000 of 8192, r = 60.
// Up to 8 components a workgroup of some 256 entries is little more than its start and end, and eight of them to a row of
// fewer than FU_XCD_ROW_FEW lose where a row makes three even chunks or fewer: 1061 / 1141 at 4000 of 2000, r = 4 (one
// chunk), 696 / 732 at 2000 of 2048, r = 8 (two), 427 / 435 at 1000 of 2200, r = 4 (three); but 1361 / 1078 at 4000 of 1800,
// r = 8 (the second chunk has 8 entries), 774 / 741 at 2000 of 2100, 511 / 475 at 1000 of 2400, 1899 / 1367 at 4000 of 2600.
static bool xcd_rows_suit(int64_t n, int64_t nnz, int r) {
  const int64_t mean = nnz / n;
  if (r > FU_XCD_RANK || mean < FU_XCD_ROW) return false;
  if (r > 8 || mean >= FU_XCD_ROW_FEW) return true;
  const int64_t chunk = fu_chunk_entries(nnz), cut = ceil_div(mean, chunk);
  return cut > 3 || 10 * mean < 9 * cut * chunk;
}
static bool by_xcd(const dnpeff_csr* S, int r) { return S->fused.x_seg && xcd_rows_suit(S->n_rows, S->nnz, r); }

// How evenly the lists deal the entries out.  out[10 workgroup + x]: entries of XCD x, + 8: the sum of the rows' largest
// shares, + 9: the largest share of all.
constexpr int FU_BALANCE = 10;
__global__ void __launch_bounds__(256) k_fu_xcd_balance(const int64_t* __restrict__ x_seg, int64_t n, unsigned long long* __restrict__ out) {
  __shared__ unsigned long long of_wave[4][FU_BALANCE];
  unsigned long long mine[FU_BALANCE] = {};
  for (int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x; row < n; row += (int64_t)gridDim.x * 256) {
    unsigned long long most = 0;
#pragma unroll
    for (int x = 0; x < 8; x++) {
      const unsigned long long len = (unsigned long long)(x_seg[8 * row + x + 1] - x_seg[8 * row + x]);
      mine[x] += len;
      most = len > most ? len : most;
    }
    mine[8] += most;
    mine[9] = most > mine[9] ? most : mine[9];
  }
  // (by shuffles: 64 lanes that meet in one LDS word ten times took 25 us at 300 rows, now 4)
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < FU_BALANCE; i++) {
      const unsigned long long other = __shfl_xor(mine[i], off);
      mine[i] = i < 9 ? mine[i] + other : other > mine[i] ? other : mine[i];
    }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < FU_BALANCE; i++) of_wave[threadIdx.x >> 6][i] = mine[i];
  __syncthreads();
  if (threadIdx.x < FU_BALANCE) {
    unsigned long long total = 0;
    for (int w = 0; w < 4; w++) {
      const unsigned long long v = of_wave[w][threadIdx.x];
      total = threadIdx.x < 9 ? total + v : v > total ? v : total;
    }
    out[FU_BALANCE * blockIdx.x + threadIdx.x] = total;
  }
}

// Column ids that repeat with a period of 128, or rows of blocks of columns, leave an XCD or a workgroup with more than
// its share, and the rest of the chip waits for it.  Ten iterations in chunks of whole rows / by XCD at 500 rows of 4096, r = 8,
// 2000 of 2048, r = 32, and 300 of 16,384, r = 32, where one XCD has 1.2 times its share: 418 / 440, 1226 / 1031, 1483 / 1058
// us, 1.4 times: 420 / 456, 1217 / 1046, 1471 / 1117, twice: 421 / 508, 1208 / 1150, 1464 / 1258, all: 391 / 976, 902 /
// 2401, 999 / 2860; where every row gives another XCD 1.6 times its share: 420 / 453, 1222 / 1039, 1490 / 1073, twice: 419 /
// 462, 1220 / 1062, 1462 / 1154, all: 421 / 684, 935 / 1646, 1034 / 2438.
static int fused_xcd_balanced(const int64_t* x_seg, int64_t n, int64_t nnz, bool* even) {
  unsigned long long* words = nullptr;
  DN_TRY(host_words(&words));
  const int wgs = (int)std::min<int64_t>(HOST_WORDS / FU_BALANCE, ceil_div(n, 256));
  hipLaunchKernelGGL(k_fu_xcd_balance, dim3((unsigned)wgs), dim3(256), 0, stream(), x_seg, n, words);
  DN_LAUNCH_CHECK();
  DN_HIP(hipStreamSynchronize(stream()));
  double xcd[8] = {}, rows = 0.0, share = 0.0, most = 0.0;
  for (int w = 0; w < wgs; w++) {
    for (int x = 0; x < 8; x++) xcd[x] += (double)words[FU_BALANCE * w + x];
    rows += (double)words[FU_BALANCE * w + 8];
    share = std::max(share, (double)words[FU_BALANCE * w + 9]);
  }
  for (double x : xcd) most = std::max(most, x);
  const double eighth = (double)nnz / 8.0;
  *even = most <= 1.25 * eighth && rows <= 1.6 * eighth && share <= 4.0 * eighth / (double)n;
  return 0;
}

static int fused_xcd_build(dnpeff_csr* S) {
  fused_plan& f = S->fused;
  const int64_t n = S->n_rows, mean = S->nnz / n;
  f.x_parts = -1;
  if (!xcd_round_robin()) return 0;
  std::vector<int64_t> rowptr((size_t)n + 1);
  DN_HIP(copy_down(rowptr.data(), S->rowptr, sizeof(int64_t) * rowptr.size()));
  int64_t most = 0;
  for (int64_t i = 0; i < n; i++) most = std::max(most, rowptr[i + 1] - rowptr[i]);
  const int64_t parts = std::max<int64_t>(1, S->nnz / (8 * n) / fu_chunk_entries(S->nnz));
  if (most > 2 * mean || 8 * n * parts >= ((int64_t)1 << 24)) return 0;
  dbuf<int32_t> col;
  dbuf<int64_t> seg;
  dbuf<float> val;
  dbuf<int> base;
  if (col.alloc(S->nnz) || val.alloc(S->nnz) || seg.alloc(8 * n + 1) || base.alloc(n + 1)) {  // (no room: chunks of whole rows)
    clear_error();
    return 0;
  }
  hipLaunchKernelGGL(k_fu_xcd_split, dim3((unsigned)n), dim3(256), 0, stream(), S->rowptr, S->colind, S->vals, n, (int)parts, col.p,
                     val.p, seg.p, base.p);
  DN_LAUNCH_CHECK();
  bool even = false;
  DN_TRY(fused_xcd_balanced(seg.p, n, S->nnz, &even));
  if (tuning().verbose != 0.0)
    fprintf(stderr, "dnpeff: A H^T %s\n", even ? "by XCD" : "in chunks of whole rows: the columns load the XCDs unevenly");
  if (!even) return 0;
  f.x_seg = seg.release();
  f.x_col = col.release();
  f.x_val = val.release();
  f.x_base = base.release();
  f.x_parts = (int)parts;
  return 0;
}

int fused_plan_build(dnpeff_csr* S, int r, bool xcd) {
  fused_plan& f = S->fused;
  hipStream_t st = stream();
  if (!f.pairs) {
    DN_CHECK(S->colptr && S->n_cols > 0, "matrix has no transposed copy");
    const int64_t groups = ceil_div(S->n_cols, FU_GROUP);
    DN_TRY(dmalloc(&f.pairs, S->nnz + 1));
    const int64_t split = std::max<int64_t>(1, std::min<int64_t>(32, 16384 / groups));
    hipLaunchKernelGGL(k_fu_pack_entries, dim3((unsigned)std::min<int64_t>(groups, 1 << 20), (unsigned)split), dim3(256), 0, st,
                       S->colptr, S->rowind, S->tvals, S->n_cols, groups, f.pairs);
    DN_LAUNCH_CHECK();
  }
  DN_TRY(fused_tiles_build(S, r));
  if (xcd && f.x_parts == 0 && S->n_panels == 0 && xcd_rows_suit(S->n_rows, S->nnz, r)) {
    DN_CHECK(has_row_major(S), "row-major copy of the matrix was released");
    DN_TRY(fused_xcd_build(S));
  }
  if (!f.chunks && !(xcd && by_xcd(S, r)) && S->n_panels == 0) {
    DN_CHECK(has_row_major(S), "row-major copy of the matrix was released");
    const int64_t chunk = fu_chunk_entries(S->nnz);
    dbuf<int64_t> base;
    DN_TRY(base.alloc(S->n_rows + 1));
    unsigned long long* host = nullptr;
    DN_TRY(host_words(&host));
    int64_t* total = reinterpret_cast<int64_t*>(host);
    DN_TRY(scan_row_chunks(S->rowptr, chunk, S->n_rows, base, total));
    DN_HIP(hipStreamSynchronize(st));
    f.n_chunks = *total;
    DN_TRY(dmalloc(&f.chunks, f.n_chunks));
    DN_TRY(dmalloc(&f.n_base, S->n_rows + 1));
    hipLaunchKernelGGL(k_fu_make_chunks, dim3((unsigned)ceil_div(S->n_rows + 1, 256)), dim3(256), 0, st, S->rowptr,
                       S->n_rows, chunk, base.p, f.chunks, f.n_base);
    DN_LAUNCH_CHECK();
  }
  return 0;
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
template <int Q_, int R_>
struct fu_tag {
  static constexpr int Q = Q_, R = R_;
};

template <class F>
static int fu_dispatch(int r, F&& f) {
  int q = r / 16, rem = (r % 16 + 3) / 4;
  if (rem == 4) q++, rem = 0;
  switch (4 * q + rem) {
#define DN_FU(Q, R) \
  case 4 * Q + R: return f(fu_tag<Q, R>{});
    DN_FU(0, 1) DN_FU(0, 2) DN_FU(0, 3)
    DN_FU(1, 0) DN_FU(1, 1) DN_FU(1, 2) DN_FU(1, 3)
    DN_FU(2, 0) DN_FU(2, 1) DN_FU(2, 2) DN_FU(2, 3)
    DN_FU(3, 0) DN_FU(3, 1) DN_FU(3, 2) DN_FU(3, 3)
    DN_FU(4, 0)
#undef DN_FU
  }
  DN_CHECK(false, "rank %d has no fused step", r);
}

int fused_gram_floats(int r) { return fu_pairs((r + 15) / 16) * 256; }
static int fu_blocks_of(int r) { return (r + 15) / 16; }

using fu_h_kernel = void (*)(const fu_tile*, int, const int64_t*, const uint2*, int, const float*, float*, float,
                             const float*, int, float*);

// Whether the Gram sums of a tile are added up in fp64: fp32 sums over all tiles of a workgroup lose what follows
// a column with large entries (W update at 2000 x 6.4 M, r = 16: error 3.3e-6, with fp64 totals 1e-7, in the same
// time).  Up to 16 components always.  Up to 32 where a workgroup has more than one tile: the totals leave room
// for four workgroups per CU instead of five, which one tile each would notice (300 x 146k, r = 20: 21.8 against
// 19.6 us) and has no use for.  Above, the registers hold the fp32 sums only.
template <int Q, int R, bool PAST>
static fu_h_kernel fu_h_of(int tile_cols, bool totals) {
  constexpr int NB = fu_blocks(Q, R);
  if constexpr (NB == 1) return tile_cols == 256 ? k_fu_h<Q, R, 4, true, PAST> : k_fu_h<Q, R, 1, true, PAST>;
  else if constexpr (NB == 2)
    return totals ? (tile_cols == 128 ? k_fu_h<Q, R, 2, true, PAST> : k_fu_h<Q, R, 1, true, PAST>)
                  : (tile_cols == 128 ? k_fu_h<Q, R, 2, false, PAST> : k_fu_h<Q, R, 1, false, PAST>);
  else return k_fu_h<Q, R, 1, false, PAST>;
}
template <int Q, int R>
static fu_h_kernel fu_h_of(int64_t m, int tile_cols, bool totals) {
  return 64 * m * fu_blocks(Q, R) <= FU_PAST_BYTES ? fu_h_of<Q, R, true>(tile_cols, totals) : fu_h_of<Q, R, false>(tile_cols, totals);
}

int fused_state::create(const dnpeff_csr* S, int64_t n, int rank, bool xcd_lists) {
  r = rank;
  xcd = xcd_lists;
  S_floats = fused_gram_floats(r);
  const fused_plan& f = S->fused;
  int64_t most = 0;  // workgroups that the chip holds
  auto count = [&]() {
    int per_cu = 0;
    if (r > FUSED_NARROW_RANK) DN_TRY(fuw_per_cu(r, &per_cu));
    else DN_TRY(fu_dispatch(r, [&](auto tag) {
      DN_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &per_cu, fu_h_of<decltype(tag)::Q, decltype(tag)::R>(S->n_cols, f.tile_cols, h_totals), 256, 0));
      return 0;
    }));
    most = (int64_t)n_cus() * (per_cu > 0 ? per_cu : 1);
    return 0;
  };
  DN_TRY(count());
  if (f.n_tiles > most) {
    h_totals = true;
    DN_TRY(count());
  }
  h_wgs = (int)(f.n_tiles < most ? f.n_tiles : most);
  // (above 32 the sums stay fp32 in registers: as many rounds of workgroups as keep them short.  3.4 M columns
  // at r = 128: in one round of 512 workgroups H^T H costs the W update an error of 8.5e-7, in four 2.0e-7; the
  // update takes 1.78 ms either way, the sum of the parts 28 against 8 us)
  if (fu_blocks_of(r) > 2) {
    const int64_t per_wg = ceil_div(f.n_tiles * f.tile_cols, h_wgs);
    h_wgs *= (int)std::max<int64_t>(ceil_div(per_wg, FU_MOST_COLS), r > FUSED_NARROW_RANK && per_wg > FU_MOST_COLS / 2 ? 2 : 1);
  }
  w_wgs = (int)ceil_div(n, r > FUSED_NARROW_RANK ? FUW_COLS : FU_ROWS_WG);
  DN_TRY(dmalloc(&gh_part, (int64_t)h_wgs * S_floats));
  DN_TRY(dmalloc(&gw_part, (int64_t)w_wgs * S_floats));
  DN_TRY(dmalloc(&gh_sum, S_floats));
  DN_TRY(dmalloc(&gw_sum, S_floats));
  DN_TRY(dmalloc(&dots, ceil_div(n, 16)));
  return 0;
}

void fused_state::destroy() {
  dfree(gh_part); dfree(gw_part); dfree(gh_sum); dfree(gw_sum); dfree(dots); dfree(n_part);
  *this = fused_state();
}

static int fu_sum(const float* part, int n_parts, int S, float* out) {
  hipLaunchKernelGGL(k_fu_sum, dim3((unsigned)(S / 16)), dim3(256), 0, stream(), part, n_parts, S, out);
  DN_LAUNCH_CHECK();
  return 0;
}

int fused_state::gram_of(const float* X, int64_t rows, bool of_h) {
  const int parts = of_h ? h_wgs : w_wgs;
  float* out = of_h ? gh_part : gw_part;
  const int64_t per = ceil_div(ceil_div(rows, parts), 64) * 64;
  const dim3 grid((unsigned)parts), block(256);
  switch (fu_blocks_of(r)) {  // (workgroups past the last row leave zeros)
#define DN_FU_GRAM(NB, K) \
  case NB: hipLaunchKernelGGL(K<NB>, grid, block, 0, stream(), X, rows, per, r, out); break;
    DN_FU_GRAM(1, k_fu_gram) DN_FU_GRAM(2, k_fu_gram) DN_FU_GRAM(3, k_fu_gram) DN_FU_GRAM(4, k_fu_gram)
    DN_FU_GRAM(5, k_fu_gram_wide) DN_FU_GRAM(6, k_fu_gram_wide) DN_FU_GRAM(7, k_fu_gram_wide) DN_FU_GRAM(8, k_fu_gram_wide)
#undef DN_FU_GRAM
    default: DN_CHECK(false, "rank %d has no fused step", r);
  }
  DN_LAUNCH_CHECK();
  (of_h ? gh_state : gw_state) = PARTS;
  return 0;
}

int fused_state::product_n(const dnpeff_csr* S, const float* H) {
  const fused_plan& f = S->fused;
  n_by_xcd = xcd && by_xcd(S, r);
  DN_CHECK(n_by_xcd || (has_row_major(S) && f.chunks), "row-major copy of the matrix was released");
  const int64_t chunks = n_by_xcd ? 8 * S->n_rows * f.x_parts : f.n_chunks;
  if (n_part_floats < chunks * r + 4) {
    dfree(n_part);
    n_part = nullptr;
    n_part_floats = chunks * r + 4;
    DN_TRY(dmalloc(&n_part, n_part_floats));
  }
  const int sums = gh_state == PARTS ? (int)ceil_div(S_floats / 16, 8) * 8 : 0;
  const dim3 grid((unsigned)(chunks + sums)), block(256);
  if (grid.x > 0) {
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, block, 0, stream(), f.chunks, f.x_seg, f.x_parts, n_by_xcd ? f.x_col : S->colind,
                         n_by_xcd ? f.x_val : S->vals, r, H, n_part, sums, gh_part, h_wgs, S_floats, gh_sum);
    };
#define DN_FU_N(LPR) n_by_xcd ? go(k_fu_n<LPR, true>) : go(k_fu_n<LPR, false>)
    if (r <= 8) DN_FU_N(2);
    else if (r <= 16) DN_FU_N(4);
    else if (r <= 32) DN_FU_N(8);
    else if (r <= 64) DN_FU_N(16);
    else DN_FU_N(32);
#undef DN_FU_N
    DN_LAUNCH_CHECK();
  }
  if (sums) gh_state = SUMMED;
  return 0;
}

bool fused_state::n_part_fits(const dnpeff_csr* S) const { return n_by_xcd == (xcd && by_xcd(S, r)); }

int fused_state::sum_h() {
  if (gh_state != PARTS) return 0;
  DN_TRY(fu_sum(gh_part, h_wgs, S_floats, gh_sum));
  gh_state = SUMMED;
  return 0;
}

int fused_state::sum_w() {
  if (gw_state != PARTS) return 0;
  DN_TRY(fu_sum(gw_part, w_wgs, S_floats, gw_sum));
  gw_state = SUMMED;
  return 0;
}

int fused_state::update_w(const dnpeff_csr* S, int64_t n, const float* Nw, float* W, float eps) {
  DN_CHECK(gh_state == SUMMED, "H^T H is not at hand");
  const float* N = Nw ? Nw : n_part;
  const int* base = Nw ? nullptr : n_by_xcd ? S->fused.x_base : S->fused.n_base;
  if (r > FUSED_NARROW_RANK)
    DN_TRY(fuw_launch_w(w_wgs, n, r, base, N, W, eps, gh_sum, gw_part));
  else DN_TRY(fu_dispatch(r, [&](auto tag) {
    hipLaunchKernelGGL((k_fu_w<decltype(tag)::Q, decltype(tag)::R>), dim3((unsigned)w_wgs), dim3(256), 0, stream(), n, r,
                       base, N, W, eps, gh_sum, 1, gw_part);
    return 0;
  }));
  DN_LAUNCH_CHECK();
  gw_state = PARTS;
  return 0;
}

int fused_state::update_h(const dnpeff_csr* S, const float* W, float* H, float eps) {
  if (gw_state == PARTS && w_wgs > fu_sum_direct(fu_blocks_of(r))) DN_TRY(sum_w());
  const float* gw = gw_state == PARTS ? gw_part : gw_sum;
  const int n_gw = gw_state == PARTS ? w_wgs : 1;
  const fused_plan& f = S->fused;
  if (r > FUSED_NARROW_RANK)
    DN_TRY(fuw_launch_h(h_wgs, f, S->colptr, r, W, H, eps, gw, n_gw, gh_part));
  else DN_TRY(fu_dispatch(r, [&](auto tag) {
    hipLaunchKernelGGL((fu_h_of<decltype(tag)::Q, decltype(tag)::R>(S->n_cols, f.tile_cols, h_totals)), dim3((unsigned)h_wgs), dim3(256), 0,
                       stream(), f.tiles, (int)f.n_tiles, S->colptr, f.pairs, r, W, H, eps, gw, n_gw, gh_part);
    return 0;
  }));
  DN_LAUNCH_CHECK();
  gh_state = PARTS;
  return 0;
}

int fused_state::loss_sums(const dnpeff_csr* S, int64_t n, const float* Nw, const float* W, double* out2) {
  DN_TRY(sum_h());
  DN_TRY(sum_w());
  const int parts = (int)ceil_div(n, 16);
  hipLaunchKernelGGL(k_fu_dot, dim3((unsigned)parts), dim3(256), 0, stream(), n, r, Nw ? nullptr : n_by_xcd ? S->fused.x_base : S->fused.n_base,
                     Nw ? Nw : n_part, W, dots);
  hipLaunchKernelGGL(k_fu_loss, dim3(1), dim3(256), 0, stream(), dots, parts, r, gw_sum, gh_sum, out2);
  DN_LAUNCH_CHECK();
  return 0;
}

double fused_tiles_bytes(int64_t m, int64_t nnz) {
  // (a group of columns is cut where its tile would pass 512 entries or more: two tiles hold more than that)
  return 16.0 * ((double)m / FUW_COLS + (double)nnz / 256.0 + 2.0);
}

double fused_list_bytes(int64_t n, int64_t m, int64_t nnz) {
  return 8.0 * (double)(nnz + 1) + fused_tiles_bytes(m, nnz) + 16.0 * (double)(FU_CHUNKS + n) + 4.0 * (double)(n + 1);
}

double fused_xcd_bytes(int64_t n, int64_t nnz, int r) {
  if (!xcd_rows_suit(n, nnz, r)) return 0.0;
  return 8.0 * (double)nnz + 68.0 * (double)(n + 1) + 4.0 * 7.0 * (double)n * r;  // (eight chunks to a row)
}

double fused_state_bytes(int64_t n, int64_t m, int64_t nnz, int r) {
  const double S = 4.0 * fused_gram_floats(r);
  // workgroups of the H update: one round of what the chip holds, or enough rounds of them
  const double wgs = (r > FUSED_NARROW_RANK ? 4.0 : 8.0) * n_cus() + ((double)m + (double)nnz / 8.0) / FU_MOST_COLS;
  return 4.0 * ((double)(FU_CHUNKS + n) * r + 4.0) + S * (wgs + (double)n / FUW_COLS + 3.0) + (double)n;
}

bool fused_supported(int64_t n, int64_t m, int64_t nnz, int r) {
  if (r > FUSED_NARROW_RANK && !use_split_bf16()) return false;
  // Rank 128 has kernels of its own for the update with its Gram matrix (k_xg_mu_gram_b16), and runs on
  // small factors are held to within 1e-5 of the two-pass path over 50 iterations, closer than two
  // ways of rounding stay to each other (both are within 2e-5 of fp64): those keep the separate kernels.  That
  // is no line of speed: ten iterations at 300 x 44,008 take 4.1 ms so and 0.88 with the fused step (0.93 at
  // r = 127), at 500 x 83,420, past the line, 1.65.
  if (r == 128 && m < 65536) return false;
  // With as many components as rows the product can become A itself: the loss is then a difference of
  // nearly equal sums whose digits depend on the order of every sum before it.  Such runs stay on the
  // kernels they have always had.
  if (r >= n) return false;
  return r >= 1 && r <= FUSED_MAX_RANK && n >= 1 && m >= 1 && nnz >= 1 && n < ((int64_t)1 << FU_ROW_BITS) &&
         n * (int64_t)r < ((int64_t)1 << 30);  // (byte offsets into W in 32 bits)
}

}  // namespace dn
