// Factorisations so small that the matrix and both factors fit the LDS of one compute unit: all iterations of a
// call in one launch of one workgroup.
//
// At this size an iteration as launches (fused.hip) is three kernels of 3 to 5 us that wait for each other, and the loss
// four more.  One workgroup of 16 waves that never leaves its LDS takes 9 us per iteration at 48 x 907 with 3,072
// entries and r = 8, bound by the issue of its vector instructions (H update 4 us, A H^T and H^T H 3, the rest of W's
// update and six barriers 2): ten iterations and the loss 117 us with the host's wait, 131 with a launch of its own for the loss
// and a wait in between, 165 as launches.
// Rows of the factors lie in LDS with their components padded to a multiple of four; lane (l % 16, l / 16) takes
// row l % 16 of a tile and its components 4 (l / 16) .. + 3, as the fp32 matrix instructions want their operands (see
// fused.hip).  An entry is its value and the byte offset of the row that it multiplies.
//
// All orders are fixed: runs repeat bit for bit, and n steps in one call give what n calls of one step give.
#include "fused.hpp"

#include <algorithm>

namespace dn {

constexpr int FS_WAVES = 16, FS_THREADS = 64 * FS_WAVES;
constexpr int64_t FS_LDS = 152 * 1024;
constexpr int FS_FIXED = 4 * (FS_WAVES * 256 + 2 * 256) + 8 * 2 * FS_WAVES;  // bytes beside what grows with the sizes

static int64_t fs_bytes(int64_t n, int64_t m, int64_t nnz, int r) {
  return FS_FIXED + 16 * (int64_t)((r + 3) / 4) * (m + 2 * n + 45) + 64 + 16 * nnz + 4 * (n + m + 2);
}

// (A column is one chain of multiply-adds: no more than 128 rows.)  Where one compute unit is slower than the launches
// the sizes are left to them: they take 145 to 160 us for ten iterations and the loss up to 128 rows, one workgroup some 47 + 0.050
// m + 0.37 n + 0.0073 nnz (500 matrices of even and of Zipf columns, 6 us off on average; with the loss in a launch of its
// own, 14 us less in the steps').  One workgroup / launches: 63 / 149
// at 8 x 40, 131 / 168 at 48 x 368 with 3,072 entries, 125 / 150 at 64 x 1000 with 1,280, 147 / 149 with 3,200; past the line
// 193 / 153 at 128 x 1000 with 6,400, 233 / 150 at 87 x 2966 with 435, 314 / 149 at 128 x 4000 with 2,560.
bool fused_small_fits(int64_t n, int64_t m, int64_t nnz, int r) {
  return r <= 16 && n <= 128 && m < 65536 && nnz < 65536 && 20 * m + 150 * n + 3 * nnz <= 40000 && fs_bytes(n, m, nnz, r) <= FS_LDS;
}

struct fs_args {
  int n, m, nnz, r, steps;
  const int64_t *rowptr, *colptr;
  const int32_t *colind, *rowind;
  const float *vals, *tvals;
  float *W, *H;
  float eps;
  double* loss;  // (or NULL) <A H^T, W>, <W^T W, H^T H> after the steps, and the ticks that these took
};

// The sum over the 16 lanes of a DPP row, in all of them.
__device__ inline float fs_row_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, true));  // row_ror:8
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, true));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x122, 0xf, 0xf, true));
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x121, 0xf, 0xf, true));
  return x;
}

__global__ void __launch_bounds__(FS_THREADS) k_fs_steps(fs_args p) {
  const long long start = wall_clock64();
  extern __shared__ __align__(16) char lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int n = p.n, m = p.m, nnz = p.nnz, r = p.r, ld = (r + 3) / 4 * 4, quads = ld / 4;
  const int m16 = (m + 15) & ~15, n16 = (n + 15) & ~15;
  double* red = reinterpret_cast<double*>(lds);                // [2][FS_WAVES]
  float* part = reinterpret_cast<float*>(red + 2 * FS_WAVES);  // [FS_WAVES][256]
  float* ga = part + FS_WAVES * 256;                           // X^T X as the A operand, and for the loss a second one
  float* H = ga + 512;                                         // [m][ld]
  float* W = H + m16 * ld;
  float* N = W + n16 * ld + 16;                                     // A H^T
  uint2* rows = reinterpret_cast<uint2*>(N + n * ld);          // entries by rows, by columns
  uint2* cols = rows + nnz;
  int* rptr = reinterpret_cast<int*>(cols + nnz);
  int* cptr = rptr + n + 1;
  auto load = [&](const float* src, float* dst, int count) {
    for (int x = tid; x < ((count + 15) & ~15) * ld; x += FS_THREADS) {
      const int i = x / ld, c = x % ld;
      dst[x] = i < count && c < r ? src[i * r + c] : 0.0f;
    }
  };
  load(p.H, H, m);
  load(p.W, W, n);
  for (int x = tid; x < nnz; x += FS_THREADS) {
    rows[x] = make_uint2(4u * (unsigned)(p.colind[x] * ld), __float_as_uint(p.vals[x]));
    cols[x] = make_uint2(4u * (unsigned)(p.rowind[x] * ld), __float_as_uint(p.tvals[x]));
  }
  for (int x = tid; x <= n; x += FS_THREADS) rptr[x] = (int)p.rowptr[x];
  for (int x = tid; x <= m; x += FS_THREADS) cptr[x] = (int)p.colptr[x];
  __syncthreads();

  const bool there = g < quads;
  const int piece = there ? 4 * g : 0;  // (lanes past the components: the first piece, not kept)
  const f32x4 zero = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // The waves' shares of X^T X (rows up to the next multiple of 16 are there, and zero).
  auto gram = [&](const float* X, int count) {
    double sum[4] = {};  // (fp32 over 16 rows at a time: a row with large entries takes bits from all that follow it)
    const float* at = X + (16 * wave + g) * ld + l16;
    for (int base = 16 * wave; base < count; base += 16 * FS_WAVES, at += 16 * FS_WAVES * ld) {
      float a[4];
      f32x4 acc = zero;
#pragma unroll
      for (int s = 0; s < 4; s++) a[s] = at[4 * s * ld];
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const float v = l16 < ld ? a[s] : 0.0f;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(v, v, acc, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) sum[i] += (double)acc[i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) part[wave * 256 + (4 * g + i) * 16 + l16] = (float)sum[i];
  };
  // Their sum in fp64: thread (lane, i) of the operand has row 4 (lane / 16) + i, column lane % 16.
  auto gram_sum = [&](float* out) {
    if (tid >= 256) return;
    const int at = (4 * (tid >> 6) + (tid & 3)) * 16 + ((tid >> 2) & 15);
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < FS_WAVES; w++) s += (double)part[w * 256 + at];
    out[tid] = (float)s;
  };
  // A H^T: a wave per row, its entries dealt to 16 lanes.
  auto product = [&]() {
    const char* Hb = reinterpret_cast<const char*>(H + piece);
    for (int i = wave; i < n; i += FS_WAVES) {
      f32x4 a = zero;
      const int e1 = rptr[i + 1];
#pragma unroll 4
      for (int e = rptr[i] + l16; e < e1; e += 16) {
        const uint2 pr = rows[e];
        const f32x4 x = *reinterpret_cast<const f32x4*>(Hb + pr.x);
#pragma unroll
        for (int c = 0; c < 4; c++) a[c] = fmaf(__uint_as_float(pr.y), x[c], a[c]);
      }
#pragma unroll
      for (int c = 0; c < 4; c++) a[c] = fs_row_sum(a[c]);
      if (l16 == 0 && there) *reinterpret_cast<f32x4*>(N + i * ld + piece) = a;
    }
  };
  // The lane's piece of its row x <- x t / (x G + eps) (padding: zero stays zero)
  auto update = [&](float* at, const f32x4& gl, const f32x4& t) {
    f32x4 x = *reinterpret_cast<const f32x4*>(at), d = zero;
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = there ? x[i] : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) d = __builtin_amdgcn_mfma_f32_16x16x4f32(gl[i], x[i], d, 0, 0, 0);
    const f32x4 q = mu_quotients(t, d + p.eps);
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = 4 * g + i < r ? x[i] * q[i] : 0.0f;
    return x;
  };

  for (int step = 0; step < p.steps; step++) {
    gram(H, m);
    product();
    __syncthreads();
    gram_sum(ga);
    __syncthreads();
    {
      const f32x4 gl = *reinterpret_cast<const f32x4*>(ga + 4 * lane);
      for (int base = 16 * wave; base < n; base += 16 * FS_WAVES) {
        const int i = base + l16;
        float* at = W + i * ld + piece;
        const f32x4 x = update(at, gl, *reinterpret_cast<const f32x4*>(N + (i < n ? i : 0) * ld + piece));
        if (i < n && there) *reinterpret_cast<f32x4*>(at) = x;
      }
    }
    __syncthreads();
    gram(W, n);
    __syncthreads();
    gram_sum(ga);
    __syncthreads();
    {
      const f32x4 gl = *reinterpret_cast<const f32x4*>(ga + 4 * lane);
      const char* Wb = reinterpret_cast<const char*>(W + piece);
      for (int base = 16 * wave; base < m; base += 16 * FS_WAVES) {
        const int j = base + l16;
        const int e0 = j < m ? cptr[j] : 0, e1 = j < m ? cptr[j + 1] : 0;
        f32x4 t[4] = {zero, zero, zero, zero};
        for (int e = e0; e < e1; e += 4) {  // (four chains)
          uint2 pr[4];
          f32x4 w[4];
#pragma unroll
          for (int u = 0; u < 4; u++) pr[u] = cols[e + u < e1 ? e + u : e];
#pragma unroll
          for (int u = 0; u < 4; u++) w[u] = *reinterpret_cast<const f32x4*>(Wb + pr[u].x);
#pragma unroll
          for (int u = 0; u < 4; u++)
            if (u == 0 || e + u < e1) {
#pragma unroll
              for (int c = 0; c < 4; c++) t[u][c] = fmaf(__uint_as_float(pr[u].y), w[u][c], t[u][c]);
            }
        }
        float* at = H + j * ld + piece;
        const f32x4 x = update(at, gl, (t[0] + t[1]) + (t[2] + t[3]));
        if (j < m && there) *reinterpret_cast<f32x4*>(at) = x;
      }
    }
    __syncthreads();
  }
  auto store = [&](const float* src, float* dst, int count) {
    for (int x = tid; x < count * r; x += FS_THREADS) dst[x] = src[x / r * ld + x % r];
  };
  if (p.steps > 0) {
    store(H, p.H, m);
    store(W, p.W, n);
  }
  if (p.loss) {
    if (tid == 0) p.loss[2] = (double)(wall_clock64() - start);
    gram(H, m);
    product();
    __syncthreads();
    gram_sum(ga);
    __syncthreads();
    gram(W, n);
    __syncthreads();
    gram_sum(ga + 256);
    __syncthreads();
    double neg = 0.0, pos = tid < 256 ? (double)ga[tid] * (double)ga[256 + tid] : 0.0;  // (zero past the rank)
    for (int x = tid; x < n * ld; x += FS_THREADS) neg += (double)N[x] * (double)W[x];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      neg += __shfl_xor(neg, off);
      pos += __shfl_xor(pos, off);
    }
    if (lane == 0) {
      red[wave] = neg;
      red[FS_WAVES + wave] = pos;
    }
    __syncthreads();
    if (tid < 2) {
      double s = 0.0;
      for (int w = 0; w < FS_WAVES; w++) s += red[tid * FS_WAVES + w];
      p.loss[tid] = s;
    }
  }
}

int fused_small_launch(const dnpeff_csr* S, int r, float* W, float* H, float eps, int steps, double* loss) {
  DN_CHECK(has_row_major(S) && S->colptr, "the matrix's arrays were released");
  fs_args p{(int)S->n_rows, (int)S->n_cols, (int)S->nnz, r, 0, S->rowptr, S->colptr, S->colind, S->rowind, S->vals, S->tvals,
            W, H, eps, loss};
  const int bytes = (int)fs_bytes(S->n_rows, S->n_cols, S->nnz, r);
  DN_HIP(hipFuncSetAttribute((const void*)k_fs_steps, hipFuncAttributeMaxDynamicSharedMemorySize, (int)FS_LDS));
  do {  // (a launch of very many steps would keep a compute unit for long)
    p.steps = std::min(steps, FUSED_SMALL_STEPS);
    hipLaunchKernelGGL(k_fs_steps, dim3(1), dim3(FS_THREADS), (size_t)bytes, stream(), p);
    DN_LAUNCH_CHECK();
    steps -= p.steps;
  } while (steps > 0);
  return 0;
}

}  // namespace dn
