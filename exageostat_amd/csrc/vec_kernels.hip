// Vector-side kernels of the likelihood: log-determinant and dot-product
// partial sums, and the rectangular matrix-vector product of kriging.
//
// Replaces, from EXAGEOSTAT_dmle_Tile (exageostat_exact/src/compute/
// MLE_dexact.c:381-399): the dmdet reduction (codelet_zmdet.c:108-139,
// core_zmdet.c:50-59) and the 1x1 CHAMELEON_dgemm_Tile dot product; from
// EXAGEOSTAT_dmle_Predict_Tile (:812-820) the dgemm C12 * alpha.
#include "common.hpp"
#include "kernels.hpp"

namespace exa {

__global__ void __launch_bounds__(256) k_logdet(TileView v, double* partial) {
  __shared__ double red[256];
  const int k = blockIdx.x;
  const double* T = tile_f64(v, k, k);
  double s = 0.0;
  for (int i = threadIdx.x; i < v.ts; i += 256) {
    const long gi = (long)k * v.ts + i;
    const double d = T[i + (long)i * v.ts];
    if (gi < v.m && d > 0.0) s += log(d);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[k] = red[0];
}

__global__ void __launch_bounds__(256) k_dot(const double* z, const double* w, long n, double* partial) {
  __shared__ double red[256];
  const long base = (long)blockIdx.x * 4096;
  double s = 0.0;
  for (int i = threadIdx.x; i < 4096; i += 256) {
    const long gi = base + i;
    if (gi < n) s += z[gi] * w[gi];
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int ww = 128; ww > 0; ww >>= 1) {
    if (threadIdx.x < ww) red[threadIdx.x] += red[threadIdx.x + ww];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// y_partial[n][row] = sum over tile column n of A(m,n)[row] x_n; one
// work-group per (tile row, 64-row block, tile column).
__global__ void __launch_bounds__(256) k_gemv_full_partial(TileView v, const double* x, double* part_out) {
  __shared__ double part[4][64];
  const int tid = threadIdx.x;
  const int r = tid & 63;
  const int g = tid >> 6;
  const int ts = v.ts;
  const int q = ts / kNB;
  const int n = blockIdx.y;
  const int m = blockIdx.x / q;
  const int rb = blockIdx.x - m * q;
  double s = 0.0;
  if (!(v.lower && n > m)) {
    const double* A = tile_f64(v, m, n) + rb * kNB + r;
    const double* xn = x + (long)n * ts;
    for (int c = g; c < ts; c += 4) s += A[(long)c * ts] * xn[c];
  }
  part[g][r] = s;
  __syncthreads();
  if (tid < 64) {
    part_out[(long)n * ((long)v.mt * ts) + (long)m * ts + rb * kNB + r] =
        (part[0][r] + part[1][r]) + (part[2][r] + part[3][r]);
  }
}

__global__ void k_sum_columns(const double* part, int ncols, long len, double* y, long m) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  double s = 0.0;
  for (int c = 0; c < ncols; ++c) s += part[(long)c * len + i];
  y[i] = s;
}

void launch_logdet(const TileView& v, double* partial, hipStream_t s) {
  hipLaunchKernelGGL(k_logdet, dim3(v.mt), dim3(256), 0, s, v, partial);
  EXA_HIP(hipGetLastError());
}

void launch_dot(const double* z, const double* w, long n, double* partial, hipStream_t s) {
  const long blocks = (n + 4095) / 4096;
  if (blocks <= 0) return;
  hipLaunchKernelGGL(k_dot, dim3((unsigned)blocks), dim3(256), 0, s, z, w, n, partial);
  EXA_HIP(hipGetLastError());
}

void launch_gemv_full_partial(const TileView& v, const double* x, double* part, hipStream_t s) {
  const int q = v.ts / kNB;
  hipLaunchKernelGGL(k_gemv_full_partial, dim3((unsigned)(v.mt * q), (unsigned)v.nt), dim3(256), 0, s, v, x,
                     part);
  EXA_HIP(hipGetLastError());
}

void launch_sum_columns(const double* part, int ncols, long len, double* y, long m, hipStream_t s) {
  hipLaunchKernelGGL(k_sum_columns, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, part, ncols, len, y, m);
  EXA_HIP(hipGetLastError());
}

// part must hold nt * mt * ts doubles.
void launch_gemv_full(const TileView& v, const double* x, double* y, double* part, hipStream_t s) {
  const int q = v.ts / kNB;
  hipLaunchKernelGGL(k_gemv_full_partial, dim3((unsigned)(v.mt * q), (unsigned)v.nt), dim3(256), 0, s, v, x,
                     part);
  const long len = (long)v.mt * v.ts;
  hipLaunchKernelGGL(k_sum_columns, dim3((unsigned)((v.m + 255) / 256)), dim3(256), 0, s, part, v.nt, len, y,
                     (long)v.m);
  EXA_HIP(hipGetLastError());
}

}  // namespace exa
