// FP64 tile Cholesky kernels: trailing update and the inverses of the
// diagonal tiles, on FP64 MFMA (the panels: chol_flow.hip).
//
// Replaces Chameleon's CHAMELEON_dpotrf_Tile(ChamLower, C) as called from
// EXAGEOSTAT_dmle_Tile (exageostat_exact/src/compute/MLE_dexact.c:372);
// Chameleon is not vendored, the algorithm is the right-looking tile
// Cholesky (potrf of A(k,k), trsm of A(m,k), syrk/gemm of A(m,n), m>=n>k).
#include "common.hpp"
#include "kernels.hpp"
#include "mfma.hpp"

#include <cstdlib>

namespace exa {

using C64 = GemmCfg<64, 64, 2, 2, 16>;

// ---------------------------------------------------------------------------
// Explicit inverse X = L_kk^-1 of every diagonal tile (for the triangular
// solves, which then become matrix-vector products).  One work-group per
// (tile k, 64-column block j): X_jj = inv(L_jj) from the potrf, then for
// i > j: X_ij = -inv(L_ii) sum_{l=j}^{i-1} L_il X_lj.
__global__ void __launch_bounds__(256) k_trtri_tiles(TileView v, const double* dinv, double* xinv) {
  __shared__ __attribute__((aligned(16))) double lds[2 * 64 * 68];
  constexpr int LDT = 68;
  const int ts = v.ts;
  const int q = ts / kNB;
  const int k = blockIdx.x / q;
  const int j = blockIdx.x - k * q;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / C64::WGN;
  const int wn = wave - wm * C64::WGN;
  const double* L = tile_f64(v, k, k);
  double* X = xinv + (long)k * ts * ts;
  const double* dk = dinv + (long)k * q * 4096;
  for (int e = tid; e < 64 * 64; e += 256) {
    const int r = e & 63, c = e >> 6;
    X[(j * kNB + r) + (long)(j * kNB + c) * ts] = dk[(long)j * 4096 + r + c * 64];
  }
  for (int e = tid; e < j * kNB * kNB; e += 256) {
    const int r = e % (j * kNB), c = e / (j * kNB);
    X[r + (long)(j * kNB + c) * ts] = 0.0;
  }
  __syncthreads();
  for (int i = j + 1; i < q; ++i) {
    dx4 acc[C64::FM][C64::FN];
    zero_acc<C64>(acc);
    gemm_nt_acc<C64, true>(acc, L + i * kNB + (long)j * kNB * ts, ts, X + j * kNB + (long)j * kNB * ts, ts,
                           (i - j) * kNB, lds, 1.0);
    double* As = lds;             // inv(L_ii): As[k][r] = inv(r, k)
    double* Bs = lds + 64 * LDT;  // acc:       Bs[k][c] = acc(k, c)
#pragma unroll
    for (int a = 0; a < C64::FM; ++a)
#pragma unroll
      for (int b = 0; b < C64::FN; ++b) {
        const int c = wn * C64::WN + b * 16 + frag_col(lane);
#pragma unroll
        for (int vv = 0; vv < 4; ++vv) {
          const int r = wm * C64::WM + a * 16 + frag_row(lane, vv);
          Bs[r * LDT + c] = acc[a][b][vv];
        }
      }
    const double* inv = dk + (long)i * 4096;
    for (int e = tid; e < 64 * 32; e += 256) {
      const int kk = e >> 5;
      const int r2 = e & 31;
      *reinterpret_cast<double2*>(As + kk * LDT + 2 * r2) = *reinterpret_cast<const double2*>(inv + 2 * r2 + kk * 64);
    }
    __syncthreads();
    dx4 y[C64::FM][C64::FN];
    zero_acc<C64>(y);
#pragma unroll 4
    for (int kk = 0; kk < 64; kk += 4) {
      const int krow = kk + (lane >> 4);
      double a[C64::FM], b[C64::FN];
#pragma unroll
      for (int ii = 0; ii < C64::FM; ++ii) a[ii] = -As[krow * LDT + wm * C64::WM + ii * 16 + (lane & 15)];
#pragma unroll
      for (int jj = 0; jj < C64::FN; ++jj) b[jj] = Bs[krow * LDT + wn * C64::WN + jj * 16 + (lane & 15)];
#pragma unroll
      for (int ii = 0; ii < C64::FM; ++ii)
#pragma unroll
        for (int jj = 0; jj < C64::FN; ++jj) y[ii][jj] = mfma_f64(a[ii], b[jj], y[ii][jj]);
    }
    acc_update<C64>(y, X + i * kNB + (long)j * kNB * ts, ts, 0.0);
    // X_ij is read back by the next i of this work-group (same CU).
    __syncthreads();
  }
}

void launch_trtri_tiles(const TileView& v, const double* dinv, double* xinv, hipStream_t s) {
  const int q = v.ts / kNB;
  hipLaunchKernelGGL(k_trtri_tiles, dim3((unsigned)(v.mt * q)), dim3(256), 0, s, v, dinv, xinv);
  EXA_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Trailing update A(m,n) -= sum_{p < np} A(m,k+p) A(n,k+p)^T over BM x BN
// blocks (np = 2: two factorisation steps at once, K = 2 ts per block and
// one read and write of C).
// Tile pairs (m, n) with n in [col_lo, col_hi] and m in [n, mt), column by
// column (consecutive pairs share the panel tile n).
//
// Persistent launch: gridDim.x work-groups (one round of the whole chip, two
// per CU; a panel on the other stream runs as they end) loop over the block
// list.  Work-groups are dispatched round-robin
// over the XCDs, so work-group w runs on XCD w % nx; each XCD gets a
// contiguous slice of the block list and its work-groups walk it together,
// which keeps the A/B row panels they share hot in that XCD's L2.
template <class C>
__device__ __forceinline__ void update_block(const TileView& v, int k, int np, int col_lo, int col_hi, long b,
                                             double* lds) {
  const int qm = v.ts / C::BM;
  const int qn = v.ts / C::BN;
  const long p = b / (qm * qn);
  const int rem = (int)(b - p * (qm * qn));
  const int bi = rem % qm;
  const int bj = rem / qm;
  // column n: the last c in [col_lo, col_hi] with pairs_before(c) <= p
  const int mt = v.mt;
  auto pairs_before = [&](int c) {
    return (long)(c - col_lo) * mt - ((long)c * (c - 1) / 2 - (long)col_lo * (col_lo - 1) / 2);
  };
  int lo = col_lo, hi = col_hi;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (pairs_before(mid) <= p) lo = mid;
    else hi = mid - 1;
  }
  const int n = lo;
  const int m = n + (int)(p - pairs_before(n));
  if (m == n && (bi + 1) * C::BM <= bj * C::BN) return;
  double* Cp = tile_f64(v, m, n) + bi * C::BM + (long)bj * C::BN * v.ts;
  dx4 acc[C::FM][C::FN];
  zero_acc<C>(acc);
  gemm_nt_pipe<C, 2>(
      acc, np,
      [&](int s, const double*& A, const double*& B) {
        A = tile_f64(v, m, k + s) + bi * C::BM;
        B = tile_f64(v, n, k + s) + bj * C::BN;
      },
      v.ts, v.ts, lds);
  pipe_sub<C>(acc, Cp, v.ts);
}

template <class C>
__global__ void __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(2))) k_tile_update(TileView v, int k, int np, int col_lo, int col_hi,
                                                      long nblocks, int nx) {
  __shared__ __attribute__((aligned(16))) double lds[PipeLds<C, 2>::DOUBLES];
  const int w = blockIdx.x;
  const int x = w % nx;
  const int gx = gridDim.x / nx;
  const long per = (nblocks + nx - 1) / nx;
  const long start = (long)x * per;
  const long end = start + per < nblocks ? start + per : nblocks;
  for (long b = start + w / nx; b < end; b += gx) update_block<C>(v, k, np, col_lo, col_hi, b, lds);
}

static int g_update_wgs = 0;

// Work-groups of the persistent update: one round of the whole chip, rounded
// down to a multiple of 8 (XCDs).  CUs kept free for the panel factorisation
// on the other stream (EXAGEOSTAT_RESERVE_CUS) cost the update more than the
// overlap gives, since a panel is one launch: with 0 / 8 / 16 of them the
// FP64 likelihood takes 49.7 / 51.5 / 52.1 ms at n = 20,000, 355 / 365 / 375 ms
// at n = 40,000 and 3.72 / 3.83 s (0 / 8) at n = 90,000.
template <class C>
static int update_grid_cap() {
  static int cap = 0;
  if (cap) return cap;
  int dev = 0, cus = 0, occ = 1;
  EXA_HIP(hipGetDevice(&dev));
  EXA_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  EXA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_tile_update<C>, C::NT, 0));
  int reserve = 0;
  if (const char* e = getenv("EXAGEOSTAT_RESERVE_CUS")) reserve = atoi(e);
  if (reserve < 0 || reserve >= cus) reserve = 0;
  cap = (cus - reserve) * (occ > 0 ? occ : 1);
  if (cap >= 8) cap -= cap % 8;
  if (cap < 1) cap = 1;
  return cap;
}

template <class C>
static void launch_update_cfg(const TileView& v, int k, int np, int col_lo, int col_hi, hipStream_t s) {
  long pairs = 0;
  for (int c = col_lo; c <= col_hi && c < v.mt; ++c) pairs += v.mt - c;
  if (pairs <= 0) return;
  const long blocks = pairs * (v.ts / C::BM) * (v.ts / C::BN);
  const int cap = update_grid_cap<C>();
  int grid = blocks < cap ? (int)blocks : cap;
  int nx = 8;
  if (grid % 8 != 0) nx = 1;
  g_update_wgs = grid;
  hipLaunchKernelGGL(k_tile_update<C>, dim3((unsigned)grid), dim3(C::NT), 0, s, v, k, np, col_lo, col_hi, blocks,
                     nx);
  EXA_HIP(hipGetLastError());
}

void launch_tile_update(const TileView& v, int k, int np, int col_lo, int col_hi, hipStream_t s) {
  if (col_hi >= v.mt) col_hi = v.mt - 1;
  if (col_lo >= v.mt || col_hi < col_lo) return;
  if (np < 1 || np > 2 || col_lo < k + np) throw std::invalid_argument("tile_update: bad panel count or columns");
  if (v.ts % 192 == 0) {
    launch_update_cfg<GemmCfg<96, 192, 2, 2, 16>>(v, k, np, col_lo, col_hi, s);
  } else if (v.ts % 128 == 0) {
    launch_update_cfg<GemmCfg<128, 128, 2, 2, 16>>(v, k, np, col_lo, col_hi, s);
  } else {
    launch_update_cfg<C64>(v, k, np, col_lo, col_hi, s);
  }
}

}  // namespace exa
