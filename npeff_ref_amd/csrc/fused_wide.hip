// The updates of the fused step at ranks 65 ... 128: as k_fu_h and k_fu_w (fused.hip), with G in
// registers.
//
// At these ranks G no longer fits LDS beside the tile, and the fp32 matrix cores would take longer than
// everything else.  X G therefore runs on the bf16 matrix cores with both operands split in three
// (split_bf16.hpp; v_mfma_f32_16x16x32_bf16, six products): a tile is 32 rows, each of the four waves
// holds the split G of its own output components in registers, and the split rows of the tile go through
// LDS.  A lane's share of X G is the layout in which it has loaded X (rows l % 16, components 16 b + 4
// (l / 16) + i), so X is read once and split by the lane that updates it.  The result is split again for
// X^T X, whose upper block pairs are dealt to the waves.
#include "fused.hpp"

namespace dn {

// The lane, of which the compiler is not told that it stays the same: what is computed from it is computed
// where it is used.  (Hoisted out of the loop over the tiles the addresses of a lane's LDS and global
// accesses took 60 registers and, at rank 128, spilled.)
__device__ inline int fuw_lane() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  return lane;
}

constexpr int FUW_U = 2;     // rows of W in flight per lane group
constexpr int FUW_RUN = 64;  // entries of a column added up one after the other
constexpr int fuw_steps(int nb) { return (16 * nb + 31) / 32; }

struct fuw_args {
  // H update
  const fu_tile* tiles;
  int n_tiles;
  const int64_t* colptr;
  const uint2* pairs;
  const float* W;
  // W update
  int64_t n;
  const int* n_base;
  const float* N;
  // both
  int r;
  float* X;
  float eps;
  const float* g;
  int n_g;
  float* gpart;
};

// Four components c .. c + 3 of a row, zero past the rank; `whole`: all of the block's exist.
__device__ inline f32x4 fuw_load4(const float* __restrict__ row, int c, int r, bool whole) {
  if (whole) return *reinterpret_cast<const f32x4u*>(row + c);
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = c + i < r ? row[c + i] : 0.0f;
  return v;
}

// Block rows of X^T X that wave W forms: W and 7 - W.  y: three planes of the split result, transposed:
// [component][32 rows], the 16-byte pieces of a component's row stored at piece ^ (component / 4 mod 4)
// (a lane writes single numbers, the four lane groups then hit different banks).
constexpr int fuw_y_plane(int nb) { return 16 * nb * FUW_COLS; }
__device__ inline int fuw_y_at(int c, int j) { return c * FUW_COLS + (((j >> 3) ^ ((c >> 2) & 3)) << 3) + (j & 7); }

template <int W, int NB>
struct fuw_gram {
  static constexpr int R2 = 7 - W;
  static constexpr bool SECOND = R2 < NB && R2 > 3;
  static constexpr int N1 = NB - W, N2 = SECOND ? NB - R2 : 0;
  struct part {
    bf16x8 h, m, l;
  };
  __device__ static inline part load(const __bf16* __restrict__ y, int b, int lane) {
    const __bf16* at = y + fuw_y_at(16 * b + (lane & 15), 8 * (lane >> 4));
    return part{*reinterpret_cast<const bf16x8*>(at), *reinterpret_cast<const bf16x8*>(at + fuw_y_plane(NB)),
                *reinterpret_cast<const bf16x8*>(at + 2 * fuw_y_plane(NB))};
  }
  __device__ static inline f32x4 mul(const part& a, const part& b, f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l, b.h, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.l, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.m, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.h, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.m, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.h, c, 0, 0, 0);
  }
  template <int NA>
  __device__ static inline void add(const __bf16* __restrict__ y, f32x4 (&acc)[NA]) {
    const int lane = fuw_lane();
    const part a = load(y, W, lane);
    part a2;
    if constexpr (SECOND) a2 = load(y, R2, lane);
#pragma unroll
    for (int b = W; b < NB; b++) {
      const part x = b == W ? a : load(y, b, lane);
      acc[b - W] = mul(a, x, acc[b - W]);
      if constexpr (SECOND) {
        if (b >= R2) acc[N1 + b - R2] = mul(a2, x, acc[N1 + b - R2]);
      }
    }
  }
  template <int NA>
  __device__ static inline void out(const f32x4 (&acc)[NA], float* __restrict__ gpart) {
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    auto put = [&](int b1, int b2, const f32x4& v) {
      float* dst = gpart + fu_pair(b1, b2, NB) * 256;
#pragma unroll
      for (int i = 0; i < 4; i++) dst[(4 * g + i) * 16 + l16] = v[i];
    };
#pragma unroll
    for (int b = W; b < NB; b++) put(W, b, acc[b - W]);
    if constexpr (SECOND) {
#pragma unroll
      for (int b = R2; b < NB; b++) put(R2, b, acc[N1 + b - R2]);
    }
  }
};

// COLS: the H update (tiles of columns, A^T W gathered); else the W update (32 rows per workgroup, the
// chunk sums of A H^T).  NB: blocks of 16 components.  Two barriers per tile: the Gram products of a
// tile run between the second one and the next tile's first, beside the rows and the gathers of the next
// tile.  1000 x 3.4 M, rank 128: 1.79 ms (matrix cores 25 % of it, vector instructions with theirs 42 %, LDS 31 %;
// 1.94 ms with the addresses kept over the loop, the descriptor asked for where it is needed
// and the rows after the Gram products).  Eight waves of 128 registers, one block each: 1.84 ms.  Infinite
// entries of X or G leave NaN (their parts are infinity and NaN), and entries below 1e-33 lose the parts that
// bf16 cannot hold.
template <int NB, bool COLS>
__global__ void __launch_bounds__(256, 2) k_fuw(const fuw_args p) {
  constexpr int NS = fuw_steps(NB), PS = 32 * NS + 8, PLANE = FUW_COLS * PS, TS = 16 * NB + 4;
  constexpr bool SPLIT_J = NB <= 6;  // two waves per 16 rows, three blocks each; else two blocks, all rows
  constexpr int BPW = SPLIT_J ? 3 : 2, JPW = SPLIT_J ? 1 : 2;
  constexpr int NA = fuw_pairs(NB);
  using Gather = fu_gather<FUW_COLS, TS, NB, 16, FUW_U>;
  constexpr int YP = fuw_y_plane(NB);
  constexpr int LDS_TILE = COLS ? 4 * (Gather::CARRY + 2048) : 0;
  extern __shared__ __align__(16) char lds[];
  float* tile = reinterpret_cast<float*>(lds);
  __bf16* planes = reinterpret_cast<__bf16*>(lds + LDS_TILE);
  __bf16* ypl = planes + 3 * PLANE;
  __shared__ int cps[2][FUW_COLS + 1];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int jb0 = SPLIT_J ? wave & 1 : 0, b0 = SPLIT_J ? 3 * (wave >> 1) : 2 * wave;
  const int r = p.r;
  const char* Wb = reinterpret_cast<const char*>(p.W);
  Gather gather;
  fu_tile_at td, nd;  // this tile and the next (a descriptor is a load that nothing else hides)
  int64_t cpv = 0;
  auto request = [&](const fu_tile_at& d) {
    gather.request(p.pairs, d);
    cpv = p.colptr[d.col0 + (tid < d.nc ? tid : d.nc)];
  };
  // The 16 lane groups share the 4096th part of all entries in a tile: 64 M entries leave 1000 to each, which
  // are not added up one after the other (H update at 2000 x 6.4 M, r = 70: error 3.2e-7, with runs 1.2e-7).
  auto gather_tile = [&]() {
    if (td.share <= FUW_RUN) gather.template run<0>(p.pairs, td, Wb, tile);
    else gather.template run<FUW_RUN>(p.pairs, td, Wb, tile);
  };
  if constexpr (COLS) {
    gather.init(r);
    td = fu_describe<Gather::NG>(p.tiles, p.n_tiles, blockIdx.x);
    nd = fu_describe<Gather::NG>(p.tiles, p.n_tiles, blockIdx.x + gridDim.x);
    request(td);
  }

  // the wave's rows of G, split: row 16 (b0 + bi) + l16, components 32 s + 8 g ..  The partial matrices come through
  // LDS in 16-byte pieces, all of a matrix under way at once; every lane picking its numbers from memory, eight at a
  // time, is a chain of trips (W update at 467 x 67 23.1 us, now 15.8, at 300 x 100 26.2 and 19.1; H update at
  // 467 x 84k, 67 components 66.8 and 64.2).  The H update of eight blocks stays with that: its loop has no register to
  // spare and spills more behind the other prologue (3.4 M columns: 1.80 ms, 1.87 with it).
  constexpr bool STAGED = !(COLS && NB == 8);
  float* stage = reinterpret_cast<float*>(lds);
  if constexpr (STAGED) {
    constexpr int S = fu_pairs(NB) * 256, Q = (S + 1023) / 1024;
    double sum[Q][4] = {};
    for (int q = 0; q < p.n_g; q++) {
      const float* src = p.g + (int64_t)q * S;
      f32x4 v[Q];
#pragma unroll
      for (int u = 0; u < Q; u++) v[u] = *reinterpret_cast<const f32x4*>(src + (1024 * u + 4 * tid < S ? 1024 * u + 4 * tid : 0));
#pragma unroll
      for (int u = 0; u < Q; u++)
#pragma unroll
        for (int i = 0; i < 4; i++) sum[u][i] += (double)v[u][i];
    }
#pragma unroll
    for (int u = 0; u < Q; u++)
      if (1024 * u + 4 * tid < S)
        *reinterpret_cast<f32x4*>(stage + 1024 * u + 4 * tid) =
            f32x4{(float)sum[u][0], (float)sum[u][1], (float)sum[u][2], (float)sum[u][3]};
    __syncthreads();
  }
  bf16x8 gh[BPW][NS], gm[BPW][NS], gl[BPW][NS];
#pragma unroll
  for (int bi = 0; bi < BPW; bi++)
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const int lane = fuw_lane(), c = 16 * (b0 + bi) + (lane & 15);
      int at[8];
#pragma unroll
      for (int t = 0; t < 8; t++) {
        const int k = 32 * s + 8 * (lane >> 4) + t, bk = k >> 4, bc = c >> 4;
        const int x = bk <= bc ? fu_pair(bk, bc, NB) * 256 + (k & 15) * 16 + (c & 15)
                               : fu_pair(bc, bk, NB) * 256 + (c & 15) * 16 + (k & 15);
        at[t] = k < r && c < r ? x : -1;
      }
      f32x4 v[2];
      if constexpr (STAGED) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
          const float w = stage[at[t] < 0 ? 0 : at[t]];
          v[t >> 2][t & 3] = at[t] < 0 ? 0.0f : w;
        }
      } else {
        double sum[8] = {};
        for (int q = 0; q < p.n_g; q++) {
          const float* src = p.g + (int64_t)q * (fu_pairs(NB) * 256);
          float w[8];
#pragma unroll
          for (int t = 0; t < 8; t++) w[t] = src[at[t] < 0 ? 0 : at[t]];
#pragma unroll
          for (int t = 0; t < 8; t++) sum[t] += (double)w[t];
        }
#pragma unroll
        for (int t = 0; t < 8; t++) v[t >> 2][t & 3] = at[t] < 0 ? 0.0f : (float)sum[t];
      }
      bf16x4 h0, m0, l0, h1, m1, l1;
      split3(v[0], h0, m0, l0);
      split3(v[1], h1, m1, l1);
      gh[bi][s] = cat8(h0, h1);
      gm[bi][s] = cat8(m0, m1);
      gl[bi][s] = cat8(l0, l1);
    }
  if constexpr (STAGED) __syncthreads();
  f32x4 acc[NA];
#pragma unroll
  for (int q = 0; q < NA; q++) acc[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // (components past the last block are never written: zeros)
  for (int x = tid; x < 3 * PLANE / 2; x += 256) reinterpret_cast<unsigned*>(planes)[x] = 0u;
  __syncthreads();

  f32x4 x[JPW][BPW], t[JPW][BPW];
  struct place {  // of a tile: its rows of X and which of the lane's it has
    float* Xb;
    int l0, nc;
  };
  auto place_of = [&](int tl) {
    place q;
    q.l0 = COLS ? td.col0 & (FUW_COLS - 1) : 0;
    const int64_t base = COLS ? td.col0 - q.l0 : (int64_t)tl * FUW_COLS;
    q.nc = COLS ? td.nc : (int)(p.n - base < FUW_COLS ? p.n - base : FUW_COLS);
    q.Xb = p.X + base * r;
    return q;
  };
  auto in_tile = [&](const place& q, int jl) { return jl >= q.l0 && jl < q.l0 + q.nc; };
  auto load_x = [&](const place& q) {
    const int lane = fuw_lane(), l16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int jp = 0; jp < JPW; jp++) {
      const int jl = 16 * (jb0 + jp) + l16;
      const float* row = q.Xb + (unsigned)(in_tile(q, jl) ? jl : q.l0) * (unsigned)r;
#pragma unroll
      for (int bi = 0; bi < BPW; bi++) {
        const int b = b0 + bi;
        if (b < NB) x[jp][bi] = fuw_load4(row, 16 * b + 4 * g, r, 16 * b + 16 <= r);
        else x[jp][bi] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
  };
  auto split_x = [&]() {
    const int lane = fuw_lane(), l16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int jp = 0; jp < JPW; jp++)
#pragma unroll
      for (int bi = 0; bi < BPW; bi++) {
        if (b0 + bi >= NB) continue;
        bf16x4 h, m, l;
        split3(x[jp][bi], h, m, l);
        __bf16* at = planes + (16 * (jb0 + jp) + l16) * PS + 16 * (b0 + bi) + 4 * g;
        *reinterpret_cast<bf16x4*>(at) = h;
        *reinterpret_cast<bf16x4*>(at + PLANE) = m;
        *reinterpret_cast<bf16x4*>(at + 2 * PLANE) = l;
      }
  };

  int tl = blockIdx.x;
  place at = place_of(tl);
  load_x(at);
  if constexpr (COLS) {
    if (tid <= at.nc) cps[0][at.l0 + tid] = (int)(cpv - td.e0);
    gather_tile();
  } else {
    const int lane = fuw_lane(), l16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int jp = 0; jp < JPW; jp++) {
      const int jl = 16 * (jb0 + jp) + l16;
      const int64_t i = (int64_t)tl * FUW_COLS + (in_tile(at, jl) ? jl : 0);
      const int k0 = p.n_base ? p.n_base[i] : (int)i, k1 = p.n_base ? p.n_base[i + 1] : (int)i + 1;
#pragma unroll
      for (int bi = 0; bi < BPW; bi++) t[jp][bi] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      for (int k = k0; k < k1; k += 4) {  // (four chunk sums under way)
        f32x4 v[4][BPW];
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
          for (int bi = 0; bi < BPW; bi++)
            v[u][bi] = b0 + bi < NB ? fuw_load4(p.N + (int64_t)(k + u < k1 ? k + u : k) * r, 16 * (b0 + bi) + 4 * g, r, 16 * (b0 + bi) + 16 <= r)
                                    : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (k + u < k1) {
#pragma unroll
            for (int bi = 0; bi < BPW; bi++) t[jp][bi] += v[u][bi];
          }
      }
    }
  }
  split_x();

  for (int par = 0;; par ^= 1) {
    const int next = tl + gridDim.x;
    const bool more = COLS && next < p.n_tiles;
    if constexpr (COLS) {
      request(nd);
    }
    __syncthreads();

    const int lane = fuw_lane(), l16 = lane & 15, g = lane >> 4;
    const float inv = 1.0f / (float)(COLS && td.share > 0 ? td.share : 1);
#pragma unroll
    for (int jp = 0; jp < JPW; jp++) {
      f32x4 d[BPW];
#pragma unroll
      for (int bi = 0; bi < BPW; bi++) d[bi] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < NS; s++) {
        const __bf16* pl = planes + (16 * (jb0 + jp) + l16) * PS + 32 * s + 8 * g;
        const bf16x8 bh = *reinterpret_cast<const bf16x8*>(pl);
        const bf16x8 bm = *reinterpret_cast<const bf16x8*>(pl + PLANE);
        const bf16x8 bl = *reinterpret_cast<const bf16x8*>(pl + 2 * PLANE);
#define DN_FUW(A, B)                            \
  _Pragma("unroll") for (int bi = 0; bi < BPW; bi++) d[bi] = \
      __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[bi][s], B, d[bi], 0, 0, 0)
        DN_FUW(gl, bh);
        DN_FUW(gh, bl);
        DN_FUW(gm, bm);
        DN_FUW(gm, bh);
        DN_FUW(gh, bm);
        DN_FUW(gh, bh);
#undef DN_FUW
      }
      const int jl = 16 * (jb0 + jp) + l16;
      const bool mine = in_tile(at, jl);
      bool some = mine;
      if constexpr (COLS) {
        const float* trow = tile + jl * TS + 4 * g;
        const int a0 = mine ? cps[par][jl] : 0, a1 = mine ? cps[par][jl + 1] : 0;
        some = a1 > a0;  // (a column without entries: 0)
#pragma unroll
        for (int bi = 0; bi < BPW; bi++)
          if (b0 + bi < NB) t[jp][bi] = *reinterpret_cast<const f32x4*>(trow + 16 * (b0 + bi));
        if (some) {
          int k0, k1;
          fu_cut_by(a0, a1, td.share, inv, k0, k1);
          for (int k = k0; k < k1; k++)
#pragma unroll
            for (int bi = 0; bi < BPW; bi++)
              if (b0 + bi < NB)
                t[jp][bi] += *reinterpret_cast<const f32x4*>(tile + Gather::CARRY + k * 128 + 16 * (b0 + bi) + 4 * g);
        }
      }
#pragma unroll
      for (int bi = 0; bi < BPW; bi++) {
        const int b = b0 + bi;
        if (b >= NB) continue;
        const bool whole = 16 * b + 16 <= r;
        f32x4 y;
        const f32x4 quot = mu_quotients(t[jp][bi], d[bi] + p.eps);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float v = x[jp][bi][i] * quot[i];
          y[i] = some ? v : 0.0f;
        }
        if (!whole) {
#pragma unroll
          for (int i = 0; i < 4; i++) y[i] = 16 * b + 4 * g + i < r ? y[i] : 0.0f;
        }
        if (mine) {
          float* dst = at.Xb + (unsigned)jl * (unsigned)r + 16 * b + 4 * g;
          if (whole) *reinterpret_cast<f32x4u*>(dst) = y;
          else {
#pragma unroll
            for (int i = 0; i < 4; i++)
              if (16 * b + 4 * g + i < r) dst[i] = y[i];
          }
        }
        bf16x4 h, m, l;
        split3(y, h, m, l);
        __bf16* yp = ypl + fuw_y_at(16 * b + 4 * g, jl);
#pragma unroll
        for (int i = 0; i < 4; i++) {  // (the four components share the piece's place)
          yp[i * FUW_COLS] = h[i];
          yp[i * FUW_COLS + YP] = m[i];
          yp[i * FUW_COLS + 2 * YP] = l[i];
        }
      }
    }
    __syncthreads();
    if (more) {
      td = nd;
      if constexpr (COLS) nd = fu_describe<Gather::NG>(p.tiles, p.n_tiles, next + gridDim.x);
      tl = next;
      at = place_of(tl);
      load_x(at);
    }
    fuw_for_wave(wave, [&](auto w) { fuw_gram<decltype(w)::value, NB>::add(ypl, acc); });
    if (!more) break;
    if constexpr (COLS) {
      if (tid <= at.nc) cps[par ^ 1][at.l0 + tid] = (int)(cpv - td.e0);
      gather_tile();
      split_x();
    }
  }
  float* out = p.gpart + (int64_t)blockIdx.x * (fu_pairs(NB) * 256);
  fuw_for_wave(wave, [&](auto w) { fuw_gram<decltype(w)::value, NB>::out(acc, out); });
}

// LDS of a workgroup of k_fuw: the tile with its carries, the split rows, the split results.
static size_t fuw_lds(int nb, bool cols) {
  const int ps = 32 * fuw_steps(nb) + 8;
  return (cols ? 4 * (size_t)(FUW_COLS * (16 * nb + 4) + 2048) : 0) + 6 * (size_t)(FUW_COLS * ps) + 6 * (size_t)fuw_y_plane(nb);
}

template <bool COLS, class F>
static int fuw_dispatch(int r, F&& f) {
  switch ((r + 15) / 16) {
    case 5: return f(k_fuw<5, COLS>);
    case 6: return f(k_fuw<6, COLS>);
    case 7: return f(k_fuw<7, COLS>);
    case 8: return f(k_fuw<8, COLS>);
  }
  DN_CHECK(false, "rank %d has no fused step", r);
}

// Dynamic LDS of more than 64 KB has to be asked for, once per kernel.
template <class K>
static int fuw_prepare(K kernel, size_t bytes) {
  DN_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return 0;
}

int fuw_per_cu(int r, int* wgs) {
  const size_t lds = fuw_lds((r + 15) / 16, true);
  DN_TRY(fuw_dispatch<true>(r, [&](auto kernel) {
    DN_TRY(fuw_prepare(kernel, lds));
    DN_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(wgs, kernel, 256, lds));
    return 0;
  }));
  return fuw_dispatch<false>(r, [&](auto kernel) { return fuw_prepare(kernel, fuw_lds((r + 15) / 16, false)); });
}

int fuw_launch_h(int wgs, const fused_plan& f, const int64_t* colptr, int r, const float* W, float* H, float eps,
                 const float* gw, int n_gw, float* gpart) {
  fuw_args p = {};
  p.tiles = f.tiles; p.n_tiles = (int)f.n_tiles; p.colptr = colptr; p.pairs = f.pairs; p.W = W;
  p.r = r; p.X = H; p.eps = eps; p.g = gw; p.n_g = n_gw; p.gpart = gpart;
  DN_TRY(fuw_dispatch<true>(r, [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(256), fuw_lds((r + 15) / 16, true), stream(), p);
    return 0;
  }));
  DN_LAUNCH_CHECK();
  return 0;
}

int fuw_launch_w(int wgs, int64_t n, int r, const int* n_base, const float* N, float* W, float eps, const float* gh,
                 float* gpart) {
  fuw_args p = {};
  p.n = n; p.n_base = n_base; p.N = N; p.r = r; p.X = W; p.eps = eps; p.g = gh; p.n_g = 1; p.gpart = gpart;
  DN_TRY(fuw_dispatch<false>(r, [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(256), fuw_lds((r + 15) / 16, false), stream(), p);
    return 0;
  }));
  DN_LAUNCH_CHECK();
  return 0;
}

}  // namespace dn
