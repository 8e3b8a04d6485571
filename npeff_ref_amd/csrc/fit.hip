// The W-only updates of the fixed-H learner, all steps of a call in one launch.
//
// W <- W * (A H^T) / (W (H H^T) + eps) works row by row, so a workgroup that holds 16 rows of W and
// of A H^T and the whole of G = H H^T can do every step of the call without touching memory in
// between: at r = 256 its registers hold G (16 columns per wave, 64 registers a lane), the 16 rows of W
// lie in LDS as the A operand of the next step (two buffers: one barrier per step) and, with A H^T, in
// registers in the accumulator layout for the update itself.  fp32 matrix cores, as the rows are too
// few for the split-operand kernels: 2,000 rows are 125 workgroups.  Bound by the matrix cores of the CUs
// it fills (16 r^2 multiply-adds per workgroup and step at 256 flop per clock and CU: 3.4 us at
// r = 256).  25 steps of 2,000 x 256: 1.22 ms as launches of a product kernel, a transposition and
// a kernel for the last rows per step; figures now at launch_fit_steps.
#include "dnpeff_internal.hpp"

#include <type_traits>

namespace dn {

typedef float acc4 __attribute__((ext_vector_type(4)));

constexpr int FIT_ROWS = 16;

// G in registers and the product of a workgroup's 16 rows (in LDS) with it.  RP: the rank padded to a
// multiple of 32; wave w owns columns 16 w .. 16 w + 15.  Lane (i = l % 16,
// kg = l / 16) reads X[row i][16 q + 4 kg .. + 3] with one 16-byte LDS read and step s of the
// group contracts component 16 q + 4 kg + s against the same row of G.
//
// A step is a chain (matrix instructions, division, LDS, barrier), so that half as many columns per wave, on twice as many
// waves, make it shorter where few waves have the chip: 25 steps and the loss at 100 x 20, the whole fit, 61 -> 54 us, 489 x
// 64 102 -> 90, 200 x 128 96 -> 91, 2000 x 256 (bound by the matrix cores) 265 -> 264.  One step of many rows: 50,000 x 50 5.0 -> 4.6
// us, x 128 14.6 -> 14.4, x 180 42.9 -> 32.9, x 256 54.4 -> 54.6; 50,000 x 90 (six waves for three) 10.2 -> 10.6, 20,000
// rows 4.2 -> 4.4, 4000 1.33 -> 1.24.
template <int RP>
struct FitTile {
  static constexpr int LD = RP + 4;  // floats per row of X in LDS
  static constexpr int Q = RP / 16, WAVES = RP / 16;
  float g[Q][4];
  int lane, wave, kg, l16;

  __device__ inline void init(const float* __restrict__ G, int r) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    l16 = lane & 15;
    kg = lane >> 4;
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int k = 16 * q + 4 * kg + s;
        const bool ok = k < r && col() < r;
        const float v = G[ok ? (int64_t)k * r + col() : 0];
        g[q][s] = ok ? v : 0.0f;
      }
  }
  __device__ inline int col() const { return 16 * wave + l16; }
  __device__ inline int row(int v) const { return 4 * kg + v; }  // of accumulator register v

  __device__ inline acc4 product(const float* buf) const {
    acc4 d = acc4{0.0f, 0.0f, 0.0f, 0.0f};
    const float* pa = buf + l16 * LD + 4 * kg;
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const float4 a = *reinterpret_cast<const float4*>(pa + 16 * q);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const float as = s == 0 ? a.x : s == 1 ? a.y : s == 2 ? a.z : a.w;
        d = __builtin_amdgcn_mfma_f32_16x16x4f32(as, g[q][s], d, 0, 0, 0);
      }
    }
    return d;
  }
};

// <A H^T, W>, <W G, W> and <WHH, W> of a lane's entries, in fp64: to the workgroup's three sums.
template <int RP>
__device__ inline void fit_sums(const FitTile<RP>& t, const float (&x)[4], const float (&ah)[4], const acc4& d, const acc4& wh,
                                double (&red)[FitTile<RP>::WAVES][3], double* __restrict__ out) {
  double s[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int v = 0; v < 4; v++) {
    s[0] += (double)ah[v] * (double)x[v];
    s[1] += (double)d[v] * (double)x[v];
    s[2] += (double)wh[v] * (double)x[v];
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s[k] += __shfl_xor(s[k], off);
    if (t.lane == 0) red[t.wave][k] = s[k];
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double sum = 0.0;
    for (int w = 0; w < FitTile<RP>::WAVES; w++) sum += red[w][threadIdx.x];
    out[threadIdx.x] = sum;
  }
}

// n_steps updates of W in place; WHH receives W G of the W before the last of them.  LOSS: the sums of k_fit_loss
// after them, bit for bit, and the ticks that the steps took, four numbers per workgroup straight to pinned memory:
// what the loss reads is at hand here, and a launch and a wait between the two are saved (a fit of 100 x 20 in 25 steps: 64 us,
// 86 before).
template <int RP, bool LOSS>
__global__ void __launch_bounds__(4 * RP)
    k_fit_steps(float* __restrict__ W, const float* __restrict__ G, const float* __restrict__ AH, float eps,
                int64_t n, int r, int n_steps, float* __restrict__ WHH, double* __restrict__ sums) {
  using T = FitTile<RP>;
  __shared__ __align__(16) float buf[2][FIT_ROWS * T::LD];
  const long long start = LOSS ? wall_clock64() : 0;
  T t;
  t.init(G, r);
  const int64_t row0 = (int64_t)blockIdx.x * FIT_ROWS;
  float x[4], ah[4];
  bool ok[4];
  int64_t at[4];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    ok[v] = row0 + t.row(v) < n && t.col() < r;
    at[v] = ok[v] ? (row0 + t.row(v)) * r + t.col() : 0;
    x[v] = W[at[v]];
    ah[v] = AH[at[v]];
  }
#pragma unroll
  for (int v = 0; v < 4; v++) {
    if (!ok[v]) x[v] = 0.0f;  // (rows and columns of the padding stay zero)
    buf[0][t.row(v) * T::LD + t.col()] = x[v];
  }
  __syncthreads();
  acc4 d;
  for (int s = 0; s < n_steps; s++) {
    d = t.product(buf[s & 1]);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const float q = ah[v] / (d[v] + eps);
      x[v] = ok[v] ? x[v] * q : 0.0f;
      buf[(s + 1) & 1][t.row(v) * T::LD + t.col()] = x[v];
    }
    __syncthreads();  // (the buffer just read is written again one barrier from here)
  }
#pragma unroll
  for (int v = 0; v < 4; v++)
    if (ok[v]) {
      W[at[v]] = x[v];
      WHH[at[v]] = d[v];
    }
  if constexpr (LOSS) {
    __shared__ double red[T::WAVES][3];
    const long long ticks = wall_clock64() - start;
    double* out = sums + (int64_t)blockIdx.x * 4;
    const acc4 now = t.product(buf[n_steps & 1]);
#pragma unroll
    for (int v = 0; v < 4; v++)
      if (!ok[v]) ah[v] = d[v] = 0.0f;
    fit_sums<RP>(t, x, ah, now, d, red, out);
    if (threadIdx.x == 0) out[3] = (double)ticks;
  }
}

// <A H^T, W>, <W G, W> and (where WHH is given) <WHH, W> of a workgroup's rows, in fp64.
template <int RP>
__global__ void __launch_bounds__(4 * RP)
    k_fit_loss(const float* __restrict__ W, const float* __restrict__ G, const float* __restrict__ AH,
               const float* __restrict__ WHH, int64_t n, int r, double* __restrict__ partials) {
  using T = FitTile<RP>;
  __shared__ __align__(16) float buf[FIT_ROWS * T::LD];
  __shared__ double red[T::WAVES][3];
  T t;
  t.init(G, r);
  const int64_t row0 = (int64_t)blockIdx.x * FIT_ROWS;
  float x[4], ah[4];
  acc4 wh;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const bool ok = row0 + t.row(v) < n && t.col() < r;
    const int64_t at = ok ? (row0 + t.row(v)) * r + t.col() : 0;
    const float w = W[at], a = AH[at], h = WHH ? WHH[at] : 0.0f;
    x[v] = ok ? w : 0.0f;
    ah[v] = ok ? a : 0.0f;
    wh[v] = ok ? h : 0.0f;
    buf[t.row(v) * T::LD + t.col()] = x[v];
  }
  __syncthreads();
  const acc4 d = t.product(buf);
  fit_sums<RP>(t, x, ah, d, wh, red, partials + (int64_t)blockIdx.x * 3);
}

// out[k] = sum of the workgroups' k-th sums, in a fixed order
__global__ void __launch_bounds__(192) k_fit_loss_sum(const double* __restrict__ partials, int64_t n_parts,
                                                      double* __restrict__ out) {
  const int k = threadIdx.x / 64, lane = threadIdx.x & 63;
  double s = 0.0;
  for (int64_t p = lane; p < n_parts; p += 64) s += partials[p * 3 + k];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (lane == 0) out[k] = s;
}

bool fit_steps_supported(int64_t n, int r) { return r >= 1 && r <= 256 && n >= 1 && n < ((int64_t)1 << 31); }
int64_t fit_loss_parts(int64_t n) { return ceil_div(n, FIT_ROWS); }

// f(integral constant RP) with the padded rank that fits r
template <class F>
static void fit_dispatch(int r, F&& f) {
  if (r <= 32) f(std::integral_constant<int, 32>{});
  else if (r <= 64) f(std::integral_constant<int, 64>{});
  else if (r <= 96) f(std::integral_constant<int, 96>{});
  else if (r <= 128) f(std::integral_constant<int, 128>{});
  else if (r <= 192) f(std::integral_constant<int, 192>{});
  else f(std::integral_constant<int, 256>{});
}

constexpr int FIT_STEPS_MAX = 256;  // per launch: 256 steps are about a millisecond per 4,096 rows at r = 256
bool fit_loss_with_steps(int64_t n, int n_steps) { return n_steps >= 1 && n_steps <= FIT_STEPS_MAX && 4 * fit_loss_parts(n) <= HOST_WORDS; }

int launch_fit_steps(int64_t n, int r, float* W, const float* G, const float* AH, float eps, int n_steps,
                     float* WHH, double* sums) {
  const dim3 grid((unsigned)ceil_div(n, FIT_ROWS));
  // (a launch of many steps would keep the device from everything else for long)
  for (int done = 0; done < n_steps; done += FIT_STEPS_MAX) {
    const int now = n_steps - done < FIT_STEPS_MAX ? n_steps - done : FIT_STEPS_MAX;
    fit_dispatch(r, [&](auto rp) {
      constexpr int RP = decltype(rp)::value;
      if (sums) hipLaunchKernelGGL((k_fit_steps<RP, true>), grid, dim3(4 * RP), 0, stream(), W, G, AH, eps, n, r, now, WHH, sums);
      else hipLaunchKernelGGL((k_fit_steps<RP, false>), grid, dim3(4 * RP), 0, stream(), W, G, AH, eps, n, r, now, WHH, sums);
    });
    DN_LAUNCH_CHECK();
  }
  return 0;
}

int launch_fit_loss(int64_t n, int r, const float* W, const float* G, const float* AH, const float* WHH,
                    double* partials, double* out3) {
  fit_dispatch(r, [&](auto rp) {
    constexpr int RP = decltype(rp)::value;
    hipLaunchKernelGGL(k_fit_loss<RP>, dim3((unsigned)ceil_div(n, FIT_ROWS)), dim3(4 * RP), 0, stream(), W, G, AH,
                       WHH, n, r, partials);
  });
  if (out3) hipLaunchKernelGGL(k_fit_loss_sum, dim3(1), dim3(192), 0, stream(), partials, fit_loss_parts(n), out3);
  DN_LAUNCH_CHECK();
  return 0;
}

}  // namespace dn
