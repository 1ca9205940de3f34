// Dataflow Cholesky: a whole range of 64-column blocks factored in one
// launch, by work-groups that claim block tasks in order and wait on
// per-row progress counters instead of on kernel boundaries.
//
// Replaces, for matrices whose factorisation is bound by its serial chain of
// panels, CHAMELEON_dpotrf_Tile(ChamLower, C) as called from
// EXAGEOSTAT_dmle_Tile (exageostat_exact/src/compute/MLE_dexact.c:372); the
// same kernel factors one tile column (diagonal tile and panel) of the
// larger matrices' right-looking tile Cholesky.
//
// Left-looking in blocks of 64: with L_il final for l < j,
//   D_j  (one task per block column j): block (j, j-1) and the diagonal:
//        L_{j,j-1} = (A_{j,j-1} - sum_l L_jl L_{j-1,l}^T) inv(L_{j-1,j-1})^T,
//        L_jj = chol(A_jj - sum_l L_jl L_jl^T), and inv(L_jj);
//   T_ij (block rows i > j+1, two or three of them per task):
//        L_ij = (A_ij - sum_l L_il L_jl^T) inv(L_jj)^T.
// A right-hand side z is one more block row (z^T above zeros): its T tasks
// turn it into (L^-1 z)^T beside the factorisation.
// The sums run as far as their operands are final and then wait for the
// next ones, so the serial chain is, per 64 columns: one 64^3 product, one
// symmetric 64^2 x 64 product, the factorisation and inverse of one 64 x 64
// block, and the hand-over to the next D task.  Everything else runs beside
// it on the other work-groups.
//
// Progress: tasks are claimed from one counter in an order in which every
// task depends on earlier ones only (D_j first in its column), and a
// work-group finishes its task before it claims another: the oldest
// unfinished task never waits on an unclaimed one, so the launch drains
// whatever share of its work-groups is resident, down to a single one.
//
// Memory: finished blocks are written through to the device's coherence
// point (agent-scope stores), then the row's counter is released at agent
// scope; a waiting work-group acquires at agent scope before it reads.
// Counters only rise.  A row's counter is stored by one task after another,
// each of which has waited for the value before (T_ij and D_j for row i at
// l = j - 1), so stores are enough there.  The diagonal's is not: D_{j+1}
// reads inv(L_jj) itself (fetch_inverse) and may store its value before D_j
// has, so both raise it (flag_raise); a plain store of D_j that arrived last
// would leave the T tasks of column j + 1 waiting for good.  A work-group
// claims, and waits for the claim, after its last counter store, so that all
// of them have arrived when it counts itself out and the last one resets.
#include "common.hpp"
#include "besselk.hpp"
#include "flow.hpp"
#include "kernels.hpp"
#include "mfma.hpp"

namespace exa {

namespace {

// Counters, one per 64 bytes.
constexpr int kClaim = 0, kExit = 16, kDiag = 32, kRows = 48;
// What a diagonal block's inverse holds before it is written: a signalling
// NaN, which no arithmetic result is.
constexpr long long kUnset = 0x7ff4dead00000001;

// x of lane N of each row of 16 lanes, in all lanes of that row.
template <int N>
__device__ __forceinline__ double row_lane(double x) {
  return __longlong_as_double(
      __builtin_amdgcn_update_dpp(0L, (long)__double_as_longlong(x), 0x150 + N, 0xf, 0xf, true));
}

// y += (x of lane N of each row of 16 lanes) * z, the broadcast inside the
// multiply-add (the compiler makes a move of its own of it: three
// instructions per pair of updates instead of two).  x must not come from
// one of the two preceding vector instructions: panel_columns waits before
// it reads the pivot, on which z depends (tests/test_flow_wait_states_cpu.py
// looks for both in the generated code).
template <int N>
__device__ __forceinline__ void fma_row_lane(double& y, double x, double z) {
  asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(y) : "v"(x), "v"(z), "n"(N));
}

// Pivots for which recip3 and rsqrt_pair hold with a margin; a panel with a
// positive one outside (subnormal, near overflow, infinite) is factored again
// by divisions and roots (diag_panel_slow).
constexpr double kPivotMin = 0x1p-1000, kPivotMax = 0x1p+1000;

// 1/y for normal y: the hardware estimate (relative error 4.7e-8 measured)
// with one third-order step, three dependent operations.
__device__ __forceinline__ double recip3(double y) {
  const double r = __builtin_amdgcn_rcp(y);
  const double e = fma(-y, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// 1/sqrt(x) and sqrt(x) for normal x > 0: the hardware estimate refined by
// two coupled Newton steps and one correction of the root.
__device__ __forceinline__ void rsqrt_pair(double x, double& rs, double& s) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  s = fma(fma(-g, g, x), h, g);
  rs = h + h;
}

// Column C's update of column C2.
template <int C, int C2>
__device__ __forceinline__ void panel_update(double (&d)[16], double (&a)[16], double nd, double na) {
  if constexpr (C2 < 16) {
    fma_row_lane<C2>(d[C2], d[C], nd);
    fma_row_lane<C2>(a[C2], d[C], na);
  }
}
template <int C, int C2>
__device__ __forceinline__ void panel_updates(double (&d)[16], double (&a)[16], double nd, double na) {
  if constexpr (C2 < 16) {
    panel_update<C, C2>(d, a, nd, na);
    panel_updates<C, C2 + 1>(d, a, nd, na);
  }
}
// The updates from column C, given -d[C] / d_c and -a[C] / d_c, with the
// chain of the next pivot's reciprocal between them: in program order, since
// the compiler does not know how long either takes.
template <int C>
__device__ __forceinline__ void panel_columns(double (&d)[16], double (&a)[16], double& own, int l16, double nd,
                                              double na) {
  if constexpr (C < 15) {
    panel_update<C, C + 1>(d, a, nd, na);
    panel_update<C, C + 2>(d, a, nd, na);
    __builtin_amdgcn_sched_barrier(0);
    // a DPP operand needs two wait states after its write, which the
    // compiler does not see inside the assembly of fma_row_lane
    asm("s_nop 1" : "+v"(d[C + 1]));
    const double piv = row_lane<C + 1>(d[C + 1]);
    __builtin_amdgcn_sched_barrier(0);
    panel_update<C, C + 3>(d, a, nd, na);
    __builtin_amdgcn_sched_barrier(0);
    const double r = __builtin_amdgcn_rcp(piv);
    __builtin_amdgcn_sched_barrier(0);
    panel_update<C, C + 4>(d, a, nd, na);
    panel_update<C, C + 5>(d, a, nd, na);
    own = l16 == C + 1 ? piv : own;
    __builtin_amdgcn_sched_barrier(0);
    const double e = fma(-piv, r, 1.0);
    __builtin_amdgcn_sched_barrier(0);
    panel_update<C, C + 6>(d, a, nd, na);
    __builtin_amdgcn_sched_barrier(0);
    const double e2 = fma(e, e, e);
    __builtin_amdgcn_sched_barrier(0);
    panel_update<C, C + 7>(d, a, nd, na);
    __builtin_amdgcn_sched_barrier(0);
    const double r3 = fma(r, e2, r);
    __builtin_amdgcn_sched_barrier(0);
    panel_update<C, C + 8>(d, a, nd, na);
    __builtin_amdgcn_sched_barrier(0);
    const double nd1 = -d[C + 1] * r3, na1 = -a[C + 1] * r3;
    __builtin_amdgcn_sched_barrier(0);
    panel_updates<C, C + 9>(d, a, nd, na);
    panel_columns<C + 1>(d, a, own, l16, nd1, na1);
  }
}
template <int C>
__device__ __forceinline__ void panel_scale(double (&d)[16], double (&a)[16], double rs) {
  if constexpr (C < 16) {
    const double r = row_lane<C>(rs);
    d[C] *= r;
    a[C] *= r;
    panel_scale<C + 1>(d, a, rs);
  }
}

// Factors a 16-column panel by one wave.  d: the 16 x 16 diagonal block, row
// i in lane i of each row of 16 lanes (all four hold a copy, so that its
// entries reach every lane by a DPP broadcast inside the row); a: 64 more
// rows, one per lane.  Square-root-free elimination
//   a_{r,c2} -= (a_rc / d_c) d_{c2,c},  d_c = d_cc,
// the columns scaled by 1/sqrt(d_c) at the end for all sixteen pivots at
// once: the dependent chain per column is a broadcast, a reciprocal, a
// product and an update.  1.13 us per panel; with v_readlane broadcasts into
// scalar registers and a square root per column 2.05 us.
// Rows below the diagonal block come out as rows of L, rows of an identity
// as rows of L^-T.  root: the diagonal entry of L of the lane's column (d
// holds it as a product, one rounding further off).  Returns the mask of
// columns whose pivot is not positive; those and all later columns are NaN
// then.  again: the first pivot outside the range that this serves is a
// positive one; the results are not to be used then.
__device__ __forceinline__ unsigned panel16(double (&d)[16], double (&a)[16], double& root, bool& again, int lane) {
  int l16 = lane & 15;
  asm("" : "+v"(l16));  // comparisons with it stay here
  double rs;
  const double piv = row_lane<0>(d[0]);
  double own = l16 == 0 ? piv : 1.0;
  const double r = recip3(piv);
  panel_columns<0>(d, a, own, l16, -d[0] * r, -a[0] * r);
  rsqrt_pair(own, rs, root);
  panel_scale<0>(d, a, rs);
  again = false;
  const unsigned odd = (unsigned)__ballot(!(own >= kPivotMin && own <= kPivotMax)) & 0xffffu;
  if (!odd) return 0;
  const unsigned bad = (unsigned)__ballot(!(own > 0.0)) & 0xffffu;
  if (__builtin_ctz(odd) < __builtin_ctz(bad | 0x10000u)) {
    again = true;
  } else {
    const int first = __builtin_ctz(bad);
#pragma unroll
    for (int c = 0; c < 16; ++c)
      if (c >= first) a[c] = d[c] = __builtin_nan("");
  }
  return bad;
}

// 16 x 16 block (bi, bj), bi >= bj, of a 64 x 64 lower matrix kept as ten
// blocks, each column-major: the fragment of four columns that a wave feeds
// to one MFMA is 64 consecutive doubles.
__device__ __forceinline__ constexpr int blk16(int bi, int bj) { return (bi * (bi + 1) / 2 + bj) * 256; }

// The diagonal fragments (bi, bj) of the 64 x 64 lower triangle by wave: the
// first block column's, which the first panel waits for, one each; the other
// six on waves 1 .. 3.
__device__ __forceinline__ int diag_count(int w) { return w == 0 ? 1 : 3; }
__device__ __forceinline__ void diag_frag(int w, int t, int& bi, int& bj) {
  // w0: (0,0); w1: (1,0) (1,1) (3,1); w2: (2,0) (2,1) (2,2); w3: (3,0) (3,2) (3,3)
  bi = w;
  bj = t;
  if (w == 1 && t == 2) {
    bi = 3;
    bj = 1;
  }
  if (w == 3 && t > 0) bj = t + 1;
}

}  // namespace

struct FlowArgs {
  TileView v;
  double* pool;   // all tiles FP64 and contiguous: the whole matrix is in range; null: one tile column only
  int k;          // that tile column
  int q;          // 64-blocks per tile side
  int j0, j1;     // block columns factored; updates from columns < j0 are already in the matrix
  int i_end;      // one past the last block row
  int j_pad;      // block columns [j1, j_pad) are padding: their inverses are the identity
  double* dinv;   // inverse of diagonal block j at dinv + 4096 j
  int* info;
  int* flags;
  double* rhs;    // one more block row, i_end: 64 x 64 blocks in sequence, its rows solved with the factor
  long long* clock;  // receives the wall clock of the start, the end, and when the last block is factored
};

namespace {

// Block row i of the matrix: its tile row and the row offset inside a tile.
struct Row {
  int m, rb;
};
__device__ __forceinline__ Row row_of(const FlowArgs& a, int i) {
  const int m = i / a.q;
  return Row{m, (i - m * a.q) * kNB};
}

// Address of the first element of block column l of a block row (tile column
// l / q, or column l - k q of tile column k).
__device__ __forceinline__ char* block_ptr(const FlowArgs& a, Row r, int l, int esize) {
  const int n = l / a.q;
  const int lc = l - n * a.q;
  const long ts = a.v.ts;
  char* tile;
  if (a.pool) tile = reinterpret_cast<char*>(a.pool) + tile_index(a.v, r.m, n) * ts * ts * 8;
  else tile = static_cast<char*>(a.v.ptr[tile_index(a.v, r.m, n)]);
  return tile + ((long)lc * kNB * ts + r.rb) * esize;
}

// Waits until the (relative) counters of four rows all exceed l and returns
// the smallest; lane t of wave 0 polls row t % 4.
__device__ __forceinline__ int wait_rows(const FlowArgs& a, int r0, int r1, int r2, int r3, int l, int* sh) {
  if (threadIdx.x < 64) {
    const int t = threadIdx.x;
    const int u = t & 3;
    const int* f = a.flags + kRows + 16 * ((u < 2 ? (u ? r1 : r0) : (u == 2 ? r2 : r3)) - a.j0);
    int got;
    for (;;) {
      got = flag_get(f);
#pragma unroll
      for (int off = 1; off < 4; off <<= 1) {
        const int o = __shfl_xor(got, off, 64);
        got = o < got ? o : got;
      }
      got = __builtin_amdgcn_readfirstlane(got);
      if (got > l) break;
      __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (t == 0) *sh = got;
  }
  __syncthreads();
  const int got = *sh;
  __syncthreads();
  return got;
}

// T tasks that are not next poll less often: all of them poll one counter
// (n = 1,600: 437 -> 407 us).
__device__ __forceinline__ void wait_diag(const FlowArgs& a, int need) {
  if (threadIdx.x == 0) {
    for (;;) {
      const int got = flag_get(a.flags + kDiag);
      if (got >= need) break;
      if (got + 1 < need) __builtin_amdgcn_s_sleep(64);
      else __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
}

// Lower blocks of the 64 x 64 inverse at src into LDS (blk16 layout).
__device__ __forceinline__ void load_inverse(const double* src, double* lds, int wave, int lane) {
#pragma unroll
  for (int t = 0; t < 5; ++t) {
    const int c = wave + 4 * t;  // 20 half blocks
    const int b = c >> 1;
    const int bi = b < 1 ? 0 : (b < 3 ? 1 : (b < 6 ? 2 : 3));
    const int bj = b - bi * (bi + 1) / 2;
    const int kk = (c & 1) * 8 + (lane >> 3);
    const int r = 2 * (lane & 7);
    const double* s = src + 16 * bi + r + (16 * bj + kk) * 64;
    __builtin_amdgcn_global_load_lds((glb_void_t*)(uintptr_t)s, (lds_void_t*)(lds + c * 128), 16, 0, 0);
  }
}

// The same from an inverse that is being written: read until no element is
// the unset value, then into LDS: one way through memory where the counter
// takes three (data written, counter set, data read).  Only the next D task
// reads like this; the counter is looked at beside it, so the loop ends in
// any case.
__device__ __forceinline__ void fetch_inverse(const FlowArgs& a, int j, double* lds, int tid) {
  const double* src = a.dinv + (long)j * 4096 + (tid & 15) + (tid >> 4) * 64;
  double v[10];
  for (int last = 0;;) {
#pragma unroll
    for (int bi = 0; bi < 4; ++bi)
#pragma unroll
      for (int bj = 0; bj <= bi; ++bj) v[bi * (bi + 1) / 2 + bj] = load_through(src + 16 * bi + 16 * bj * 64);
    bool unset = false;
#pragma unroll
    for (int t = 0; t < 10; ++t) unset |= __double_as_longlong(v[t]) == kUnset;
    if (!unset || last) break;
    // The last look follows the counter by an acquire at agent scope, which
    // pairs with its release: it sees the whole inverse.
    last = flag_get(a.flags + kDiag) > j - a.j0;
    if (last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    else __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
  __syncthreads();  // the LDS may still be read
#pragma unroll
  for (int t = 0; t < 10; ++t) lds[t * 256 + tid] = v[t];
  __syncthreads();
}

// x = -t inv^T for the wave's 16 rows: t and x are 16 x 64, four fragments of
// lane l, element v at row l%16, column 16 f + l/16 + 4 v.  That is also the
// layout in which the MFMA takes its left operand, so t feeds it as is.
__device__ __forceinline__ void times_inverse(const dx4 (&t)[4], dx4 (&x)[4], const double* inv, int lane) {
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    x[f] = dx4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int g = 0; g <= f; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[f] = mfma_f64(inv[blk16(f, g) + e * 64 + lane], -t[g][e], x[f]);
  }
}

// A stage of the operand ring: NP panels of 64 rows x 16 columns.
constexpr int kPanel = 1024;

// acc[p][f] += A_p B^T over block columns [l, l_end): A_p the block rows
// `ra` (R of them; FP32 tiles when TA is float; with RHS the right-hand
// sides' row instead), B the block row rb.
// DIAG: instead, panel 0 is block row ra[0] = j-1 and panel B is j, and
// acc[0][f] += B A^T, dacc += the wave's fragments of B B^T.
template <int R, class TA, bool DIAG, bool RHS = false>
__device__ __forceinline__ void flow_gemm(const FlowArgs& a, dx4 (&acc)[R][4], dx4 (&dacc)[3], const Row (&ra)[R],
                                          Row rb, int l, int l_end, double* lds) {
  constexpr bool kF = sizeof(TA) == 4;
  constexpr int A_PAN = kF ? kPanel / 2 : kPanel;  // doubles
  constexpr int STAGE = R * A_PAN + kPanel;
  constexpr int PER_WAVE = R * (kF ? 1 : 2) + 2;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ts = a.v.ts;
  const int nk = (l_end - l) * 4;
  if (nk <= 0) return;
  const char* pa[R];
  const char* pb = block_ptr(a, rb, l, 8);
#pragma unroll
  for (int p = 0; p < R; ++p)
    pa[p] = RHS ? reinterpret_cast<char*>(a.rhs + (long)l * 4096) : block_ptr(a, ra[p], l, (int)sizeof(TA));
  int n = l / a.q;
  int left = (a.q - (l - n * a.q)) * 4;  // slices left in the current tile column
  // byte offsets of this lane's elements in a slice
  uint32_t o8[2], o4, oz[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int kk = 4 * wave + 2 * e + (lane >> 5);
    o8[e] = (uint32_t)((((2 * (lane & 31)) ^ ((kk & 1) * 16)) + kk * ts) * 8);
    if (RHS) oz[e] = (uint32_t)((((2 * (lane & 31)) ^ ((kk & 1) * 16)) + kk * kNB) * 8);
  }
  {
    const int kk = 4 * wave + (lane >> 4);
    o4 = (uint32_t)((((4 * (lane & 15)) ^ ((kk & 3) * 16)) + kk * ts) * 4);
  }
  auto issue = [&](int buf) {
    if (left == 0) {
      ++n;
      pb = block_ptr(a, rb, n * a.q, 8);
#pragma unroll
      for (int p = 0; p < R; ++p)
        if (!RHS) pa[p] = block_ptr(a, ra[p], n * a.q, (int)sizeof(TA));
      left = a.q * 4;
    }
    double* st = lds + buf * STAGE;
#pragma unroll
    for (int p = 0; p < R; ++p) {
      if constexpr (kF) {
        __builtin_amdgcn_global_load_lds((glb_void_t*)(uintptr_t)(pa[p] + o4),
                                         (lds_void_t*)(st + p * A_PAN + wave * 128), 16, 0, 0);
      } else {
#pragma unroll
        for (int e = 0; e < 2; ++e)
          __builtin_amdgcn_global_load_lds((glb_void_t*)(uintptr_t)(pa[p] + (RHS ? oz[e] : o8[e])),
                                           (lds_void_t*)(st + p * A_PAN + (2 * wave + e) * 128), 16, 0, 0);
      }
      pa[p] += (long)16 * (RHS ? kNB : ts) * sizeof(TA);
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
      __builtin_amdgcn_global_load_lds((glb_void_t*)(uintptr_t)(pb + o8[e]),
                                       (lds_void_t*)(st + R * A_PAN + (2 * wave + e) * 128), 16, 0, 0);
    pb += (long)16 * ts * 8;
    --left;
  };
  const int k4 = lane >> 4, r16 = lane & 15;
  const int flip = (k4 & 1) * 16;
  int dbi[3], dbj[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) diag_frag(wave, t < diag_count(wave) ? t : 0, dbi[t], dbj[t]);
  double fa[2][R], fb[2][4], fx[2][3], fy[2][3];
  auto frag = [&](int set, int buf, int kk) {
    const double* st = lds + buf * STAGE;
    const int k = 4 * kk + k4;
    const double* Bp = st + R * A_PAN + k * 64 + r16;
    if constexpr (DIAG) {
      const double* Ap = st + k * 64 + r16;
      fa[set][0] = Bp[(16 * wave) ^ flip];
#pragma unroll
      for (int f = 0; f < 4; ++f) fb[set][f] = Ap[(16 * f) ^ flip];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        fx[set][t] = Bp[(16 * dbi[t]) ^ flip];
        fy[set][t] = Bp[(16 * dbj[t]) ^ flip];
      }
    } else {
#pragma unroll
      for (int p = 0; p < R; ++p) {
        if constexpr (kF) {
          const float* Af = reinterpret_cast<const float*>(st + p * A_PAN);
          fa[set][p] = (double)Af[k * 64 + ((16 * wave) ^ (k4 * 16)) + r16];
        } else {
          fa[set][p] = st[p * A_PAN + k * 64 + ((16 * wave) ^ flip) + r16];
        }
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) fb[set][f] = Bp[(16 * f) ^ flip];
    }
  };
  auto step = [&](int cur) {
#pragma unroll
    for (int p = 0; p < R; ++p)
#pragma unroll
      for (int f = 0; f < 4; ++f) acc[p][f] = mfma_f64(fb[cur][f], fa[cur][p], acc[p][f]);
    if constexpr (DIAG) {
#pragma unroll
      for (int t = 0; t < 3; ++t)
        if (t == 0 || wave != 0) dacc[t] = mfma_f64(fy[cur][t], fx[cur][t], dacc[t]);
    }
  };
  __builtin_amdgcn_s_barrier();
  issue(0);
  issue(1);  // nk >= 4
  wait_vmcnt<PER_WAVE>();
  __builtin_amdgcn_s_barrier();
  frag(0, 0, 0);
  int buf = 0;
#pragma unroll 1
  for (int kc = 0; kc < nk; ++kc) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int cur = kk & 1, nxt = cur ^ 1;
      if (kk < 3) {
        frag(nxt, buf, kk + 1);
      } else if (kc + 1 < nk) {
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt_lgkm0<0>();
        __builtin_amdgcn_s_barrier();
        if (kc + 2 < nk) issue(buf);
        frag(nxt, buf ^ 1, 0);
      }
      step(cur);
      __builtin_amdgcn_sched_barrier(0);
    }
    buf ^= 1;
  }
}

typedef __attribute__((address_space(1))) double gdouble;

// The wave's 16 rows of a 64 x 64 block.
template <class TA>
__device__ __forceinline__ void block_load(const char* blk, long ts, int wave, int lane, dx4 (&c)[4]) {
  typedef __attribute__((address_space(1))) const TA gT;
  gT* G = (gT*)(uintptr_t)blk + 16 * wave + (lane & 15) + (long)(lane >> 4) * ts;
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int v = 0; v < 4; ++v) c[f][v] = (double)G[(long)(16 * f + 4 * v) * ts];
}

// The sums of products run from zero over kSumBlocks block columns each and
// are then subtracted from C.  Added to -C one after another, every product
// would be rounded at C's magnitude, and in one long sum at that sum's: error
// of z^T C^-1 z (rms, against 80-bit arithmetic, exponential kernel, nugget 0 /
// 0.05) at n = 5,000 58e-16 / 28e-16 and at 9,000 68e-16 / 75e-16 from -C, 15e-16 /
// 8e-16 and 17e-16 / 10e-16 from zero, 7e-16 / 8e-16 and 11e-16 / 7e-16 like this; the
// time is the same.
constexpr int kSumBlocks = 16;
template <int N>
__device__ __forceinline__ void sum_zero(dx4 (&acc)[N]) {
#pragma unroll
  for (int f = 0; f < N; ++f) acc[f] = dx4{0.0, 0.0, 0.0, 0.0};
}
template <int N>
__device__ __forceinline__ void sum_flush(dx4 (&acc)[N], dx4 (&c)[N]) {
#pragma unroll
  for (int f = 0; f < N; ++f) c[f] -= acc[f];
  sum_zero(acc);
}
// acc = -(C - acc)
__device__ __forceinline__ void block_sub(dx4 (&acc)[4], const dx4 (&c)[4]) {
#pragma unroll
  for (int f = 0; f < 4; ++f) acc[f] -= c[f];
}

template <class TA>
__device__ __forceinline__ void block_store(char* blk, long ts, int wave, int lane, const dx4 (&x)[4]) {
  TA* G = reinterpret_cast<TA*>(blk) + 16 * wave + (lane & 15) + (long)(lane >> 4) * ts;
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int v = 0; v < 4; ++v) store_through(G + (long)(16 * f + 4 * v) * ts, (TA)x[f][v]);
}

// T task: block rows i0 .. i0 + nr - 1 (nr <= R), block column j.
template <int R, class TA>
__device__ __forceinline__ void task_rows(const FlowArgs& a, int i0, int nr, int j, double* lds, int* sh) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long ts = a.v.ts;
  Row ra[R];
#pragma unroll
  for (int p = 0; p < R; ++p) ra[p] = row_of(a, i0 + (p < nr ? p : 0));
  const Row rj = row_of(a, j);
  // The row that D_{j+2} waits for goes ahead of the group's others.  Its
  // counter is then D_{j+2}'s: it is not stored again with theirs.
  const bool early = i0 == j + 2 && nr > 1;
  // Two rows' C is read ahead of everything (at the end, n = 1,600 took 373 us
  // instead of 358); for three there are no registers, and it is read row by
  // row, the first during the wait for the inverse.
  constexpr int AHEAD = R < 3 ? R : 1;
  dx4 acc[R][4], c[AHEAD][4], none[3];
  auto load_c = [&](int p) {
    block_load<TA>(block_ptr(a, ra[p < R ? p : 0], j, (int)sizeof(TA)), ts, wave, lane, c[p % AHEAD]);
  };
  if constexpr (AHEAD == R) {
#pragma unroll
    for (int p = 0; p < R; ++p) load_c(p);
  }
#pragma unroll
  for (int p = 0; p < R; ++p) sum_zero(acc[p]);
  int l = a.j0, have = l, flush = l + kSumBlocks;
  while (l < j) {
    if (have <= l) have = a.j0 + wait_rows(a, j, i0, i0 + nr - 1, i0 + (nr > 1 ? 1 : 0), l - a.j0, sh);
    int upto = have < j ? have : j;
    if (AHEAD == R && upto > flush) upto = flush;
    flow_gemm<R, TA, false>(a, acc, none, ra, rj, l, upto, lds);
    l = upto;
    if (AHEAD == R && l == flush) {
#pragma unroll
      for (int p = 0; p < R; ++p) sum_flush(acc[p], c[p % AHEAD]);
      flush += kSumBlocks;
    }
  }
  if constexpr (AHEAD < R) load_c(0);
  wait_diag(a, j - a.j0 + 1);  // its barrier also ends the reads of the ring
  load_inverse(a.dinv + (long)j * 4096, lds, wave, lane);
  wait_vmcnt<0>();
  __syncthreads();
#pragma unroll
  for (int p = 0; p < R; ++p) {
    if (p < nr) {
      dx4 x[4];
      block_sub(acc[p], c[p % AHEAD]);
      if (p + AHEAD < R) load_c(p + AHEAD);
      times_inverse(acc[p], x, lds, lane);
      block_store<TA>(block_ptr(a, ra[p], j, (int)sizeof(TA)), ts, wave, lane, x);
    }
    if (p == 0 && early) {
      stores_done();
      __syncthreads();
      if (tid == 0) flag_set(a.flags + kRows + 16 * (i0 - a.j0), j - a.j0 + 1);
    }
  }
  stores_done();
  __syncthreads();
  if (tid < nr && !(early && tid == 0)) flag_set(a.flags + kRows + 16 * (i0 + tid - a.j0), j - a.j0 + 1);
}

// The T task of the right-hand sides' row.
__device__ __forceinline__ void task_rhs(const FlowArgs& a, int j, double* lds, int* sh) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Row rj = row_of(a, j);
  const Row none_row[1] = {rj};
  dx4 acc[1][4], c[4], none[3];
  char* blk = reinterpret_cast<char*>(a.rhs + (long)j * 4096);
  block_load<double>(blk, kNB, wave, lane, c);
  sum_zero(acc[0]);
  int l = a.j0, have = l, flush = l + kSumBlocks;
  while (l < j) {
    if (have <= l) have = a.j0 + wait_rows(a, j, a.i_end, j, a.i_end, l - a.j0, sh);
    int upto = have < j ? have : j;
    if (upto > flush) upto = flush;
    flow_gemm<1, double, false, true>(a, acc, none, none_row, rj, l, upto, lds);
    l = upto;
    if (l == flush) {
      sum_flush(acc[0], c);
      flush += kSumBlocks;
    }
  }
  wait_diag(a, j - a.j0 + 1);
  if (tid == 0 && j + 1 == a.j1) a.clock[2] = wall_clock64();
  load_inverse(a.dinv + (long)j * 4096, lds, wave, lane);
  wait_vmcnt<0>();
  __syncthreads();
  dx4 x[4];
  block_sub(acc[0], c);
  times_inverse(acc[0], x, lds, lane);
  block_store<double>(blk, kNB, wave, lane, x);
  stores_done();
  __syncthreads();
  if (tid == 0) flag_set(a.flags + kRows + 16 * (a.i_end - a.j0), j - a.j0 + 1);
}

// LDS of a D task (doubles): the operand ring, then X = L_{j,j-1}; the
// factor's and the inverse's 16 x 16 blocks, and a 16 x 16 identity.
constexpr int kLs = 4096, kXs = kLs + 2560, kId = kXs + 2560, kDiagLds = kId + 256;

// S(bi, bj) -= L(bi, p) L(bj, p)^T, the product summed by itself like the long
// sums
__device__ __forceinline__ void diag_update(double* Ls, int bi, int bj, int p, int lane) {
  double* S = Ls + blk16(bi, bj) + lane;
  const double* A = Ls + blk16(bi, p) + lane;
  const double* B = Ls + blk16(bj, p) + lane;
  const dx4 c = {S[0], S[64], S[128], S[192]};
  dx4 s = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int e = 0; e < 4; ++e) s = mfma_f64(B[e * 64], A[e * 64], s);
#pragma unroll
  for (int e = 0; e < 4; ++e) S[e * 64] = c[e] - s[e];
}
// y += L(p, l) X(l, b); y: lane l, element v at row l/16 + 4 v, column l%16.
__device__ __forceinline__ void inverse_sum(const double* Ls, const double* Xs, dx4& y, int p, int l, int b,
                                            int lane) {
  const double* A = Ls + blk16(p, l) + lane;
  const double* B = Xs + blk16(l, b) + (lane & 15) * 16 + (lane >> 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) y = mfma_f64(A[e * 64], B[e * 4], y);
}
// X(p, b) = -X(p, p) y, in the layout of a 16 x 16 block (element e of lane
// l at 64 e + l).
__device__ __forceinline__ dx4 inverse_of(const double* Xs, const dx4& y, int p, int lane) {
  const double* D = Xs + blk16(p, p) + lane;
  dx4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int e = 0; e < 4; ++e) x = mfma_f64(-y[e], D[e * 64], x);
  return x;
}
__device__ __forceinline__ void inverse_put(double* Xs, const dx4& y, int p, int b, int lane) {
  const dx4 x = inverse_of(Xs, y, p, lane);
  double* dst = Xs + blk16(p, b) + lane;
#pragma unroll
  for (int e = 0; e < 4; ++e) dst[e * 64] = x[e];
}

// The wave's LDS accesses before it are done, and seen by all its lanes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Panel p of the diagonal block, by one wave, in LDS and with a root and
// divisions per column: for pivots at the ends of the range of doubles and
// infinite ones (whose column becomes zero), which diag_panel's reciprocals
// do not serve.  Rare, so its time does not matter.
__device__ __forceinline__ void diag_panel_slow(const FlowArgs& a, int j, int p, double* Ls, double* Xs, int lane) {
  asm("" : "+v"(lane));  // nothing of this is computed ahead of its call
  double* D = Ls + blk16(p, p);
  const int bi = p + (lane >> 4);
  // the lane's row of 16, step apart: of an identity (lanes 0 .. 15, in Xs) or
  // of a block row below
  double* row = lane < 16 ? Xs + blk16(p, p) + 16 * lane : Ls + blk16(bi < 4 ? bi : p, p) + (lane & 15);
  const int step = lane < 16 ? 1 : 16;
  const bool mine = bi < 4;
  if (lane < 16)
    for (int e = 0; e < 16; ++e) row[e] = e == lane ? 1.0 : 0.0;
  wave_sync();
#pragma unroll 1
  for (int c = 0; c < 16; ++c) {
    const double piv = D[c * 16 + c];
    const bool bad = !(piv > 0.0);
    if (bad && lane == 0) atomicCAS(a.info, 0, j * kNB + 16 * p + c + 1);
    const double s = bad ? __builtin_nan("") : sqrt(piv);
    wave_sync();
    if (lane < 16 && lane >= c) D[c * 16 + lane] = lane > c ? D[c * 16 + lane] / s : s;
    if (mine) row[c * step] /= s;
    wave_sync();
#pragma unroll 1
    for (int e = c + 1; e < 16; ++e) {
      const double l = D[c * 16 + e];
      if (lane < 16 && lane >= e) D[e * 16 + lane] -= D[c * 16 + lane] * l;
      if (mine) row[e * step] -= row[c * step] * l;
    }
    wave_sync();
  }
}

// Panel p of the diagonal block, by one wave.
__device__ __forceinline__ void diag_panel(const FlowArgs& a, int j, int p, double* Ls, double* Xs, const double* id,
                                           int lane) {
  // lanes 0 .. 15 of c: an identity (its rows become the inverse's columns);
  // 16 .. 63: block rows p + 1 ..
  double d[16], c[16];
  const int l16 = lane & 15, bi = p + (lane >> 4);
  const double* dd = Ls + blk16(p, p) + l16;
  const double* cc = (lane < 16 ? id : Ls + blk16(bi < 4 ? bi : p, p)) + l16;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    d[e] = dd[e * 16];
    c[e] = cc[e * 16];
  }
  double root;
  bool again;
  const unsigned bad = panel16(d, c, root, again, lane);
  if (again) {
    diag_panel_slow(a, j, p, Ls, Xs, lane);
    return;
  }
  if (bad && lane == 0) atomicCAS(a.info, 0, j * kNB + 16 * p + __builtin_ctz(bad) + 1);
  if (lane < 16) {
    double* dst = Xs + blk16(p, p) + lane * 16;
    double* ldst = Ls + blk16(p, p) + lane;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dst[e] = c[e];
      ldst[e * 16] = d[e];  // the zeros above the diagonal when it is written out
    }
    if (!(bad & ((2u << lane) - 1))) ldst[lane * 16] = root;  // (from the first bad column on: the NaN)
  } else if (bi < 4) {
    double* dst = Ls + blk16(bi, p) + l16;
#pragma unroll
    for (int e = 0; e < 16; ++e) dst[e * 16] = c[e];
  }
}

// D task of block column j.  After the hand-over from D_{j-1}: X = L_{j,j-1},
// S = A_jj - sum L L^T, then four 16-column panels of S by wave 0, while
// waves 1 .. 3 bring the blocks that the next panels need up to date and
// build the inverse; block row bi of S and of the inverse's sums stays with
// wave bi.
// Measured per block column (n = 1,600): 14.3 us, of which 9.0 are the four
// panels and what lies between them, 1.7 X, 1.2 the first fragments and the
// stores of X, 0.6 the last row of the inverse, 1.7 its way into the next
// task's LDS; 17.0 before the hand-over read the inverse itself
// (fetch_inverse), X was published ahead of the panels, the blocks that the
// sums are subtracted from were read ahead, and the waiting T tasks polled less.
__device__ __forceinline__ void task_diag(const FlowArgs& a, int j, double* lds, int* sh) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long ts = a.v.ts;
  const Row rj = row_of(a, j);
  const int nd = diag_count(wave);
  __builtin_amdgcn_s_setprio(2);
  double* Ls = lds + kLs;
  double* Xs = lds + kXs;
  dx4 acc[1][4], dacc[3], cx[4], dc[3];
  char* cjj = block_ptr(a, rj, j, 8);
  const bool chained = j > a.j0;
  char* cp = nullptr;
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    int bi, bj;
    diag_frag(wave, t < nd ? t : 0, bi, bj);
    gdouble* G = (gdouble*)(uintptr_t)cjj + 16 * bi + (lane & 15) + (long)(16 * bj + (lane >> 4)) * ts;
#pragma unroll
    for (int v = 0; v < 4; ++v) dc[t][v] = G[(long)(4 * v) * ts];
  }
  sum_zero(dacc);
  if (chained) {
    cp = block_ptr(a, rj, j - 1, 8);
    block_load<double>(cp, ts, wave, lane, cx);
    sum_zero(acc[0]);
    const Row rp[1] = {row_of(a, j - 1)};
    int l = a.j0, have = l, flush = l + kSumBlocks;
    while (l < j - 1) {
      if (have <= l) have = a.j0 + wait_rows(a, j, j - 1, j, j - 1, l - a.j0, sh);
      int upto = have < j - 1 ? have : j - 1;
      if (upto > flush) upto = flush;
      flow_gemm<1, double, true>(a, acc, dacc, rp, rj, l, upto, lds);
      l = upto;
      if (l == flush) {
        sum_flush(acc[0], cx);
        sum_flush(dacc, dc);
        flush += kSumBlocks;
      }
    }
    block_sub(acc[0], cx);
  }
  // S's fragment t: minus X X^T when there is one, into LDS
  auto s_frag = [&](int t) {
    int bi, bj;
    diag_frag(wave, t, bi, bj);
    if (chained) {
      const double* X = lds + bi * 1024 + lane;
      const double* Y = lds + bj * 1024 + lane;
#pragma unroll
      for (int e = 0; e < 16; ++e) dacc[t] = mfma_f64(Y[e * 64], X[e * 64], dacc[t]);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) Ls[blk16(bi, bj) + v * 64 + lane] = dc[t][v] - dacc[t][v];
  };
  if (chained) {
    fetch_inverse(a, j - 1, Xs, tid);
    dx4 x[4];
    times_inverse(acc[0], x, Xs, lane);
    // X as sixteen 16 x 16 blocks (row block w, column block f), for X X^T
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int v = 0; v < 4; ++v) lds[(wave * 4 + f) * 256 + v * 64 + lane] = x[f][v];
    block_store<double>(cp, ts, wave, lane, x);
  }
  __syncthreads();
  s_frag(0);
  stores_done();
  __syncthreads();
  // X is out: D_{j+1} and the T tasks of its column wait for it
  if (chained && tid == 64) flag_set(a.flags + kRows + 16 * (j - a.j0), j - a.j0);
  if (wave == 0) {
    diag_panel(a, j, 0, Ls, Xs, lds + kId, lane);
  } else {
    s_frag(1);
    s_frag(2);
  }
  __syncthreads();
  if (wave > 0) diag_update(Ls, wave, 1, 0, lane);
  __syncthreads();
  dx4 y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
  for (int p = 1; p < 4; ++p) {
    if (wave == 0) {
      diag_panel(a, j, p, Ls, Xs, lds + kId, lane);
    } else {
      // what panel p - 1 leaves for the panels after p, and the inverse
      for (int bj = p + 1; bj <= wave; ++bj) diag_update(Ls, wave, bj, p - 1, lane);
      if (p == 2 && wave == 1) {
        dx4 z = {0.0, 0.0, 0.0, 0.0};
        inverse_sum(Ls, Xs, z, 1, 0, 0, lane);
        inverse_put(Xs, z, 1, 0, lane);
      }
      if (p == 3 && wave < 3) {
        const int b = wave - 1;
        dx4 z = {0.0, 0.0, 0.0, 0.0};
        for (int l = b; l < 2; ++l) {
          inverse_sum(Ls, Xs, z, 2, l, b, lane);
          inverse_sum(Ls, Xs, y, 3, l, b, lane);
        }
        inverse_put(Xs, z, 2, b, lane);
      }
    }
    __syncthreads();
    if (p == 3) break;
    if (wave > p) diag_update(Ls, wave, p + 1, p, lane);
    __syncthreads();
  }
  // the inverse, then the counter that every T task of this column waits
  // for; the last block row straight from the registers of waves 1 .. 3
  double* dinv = a.dinv + (long)j * 4096;
  if (wave > 0) {
    inverse_sum(Ls, Xs, y, 3, 2, wave - 1, lane);
    const dx4 x = inverse_of(Xs, y, 3, lane);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      store_through(dinv + 48 + (lane & 15) + (16 * (wave - 1) + 4 * e + (lane >> 4)) * 64, x[e]);
  }
  const int r = tid & 15, c = tid >> 4;
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
#pragma unroll
    for (int bj = bi == 3 ? 3 : 0; bj <= bi; ++bj)
      store_through(dinv + 16 * bi + r + (16 * bj + c) * 64, Xs[blk16(bi, bj) + tid]);
  stores_done();
  __syncthreads();
  if (tid == 0) flag_raise(a.flags + kDiag, j - a.j0 + 1);
  __builtin_amdgcn_s_setprio(0);
  // off the chain: the factor block itself, the zeros above it
  gdouble* out = (gdouble*)(uintptr_t)cjj;
#pragma unroll
  for (int bi = 0; bi < 4; ++bi)
#pragma unroll
    for (int bj = 0; bj < 4; ++bj) {
      out[16 * bi + r + (long)(16 * bj + c) * ts] =
          bj < bi || (bj == bi && r >= c) ? Ls[blk16(bi, bj <= bi ? bj : 0) + tid] : 0.0;
      if (bj > bi) dinv[16 * bi + r + (16 * bj + c) * 64] = 0.0;
    }
  gdouble* top = out - rj.rb;
  for (int e = tid; e < rj.rb * kNB; e += 256) {
    const int cc = e / rj.rb;
    top[e - cc * rj.rb + (long)cc * ts] = 0.0;
  }
  __syncthreads();
}

// The T tasks of one block column: groups of up to R consecutive block rows
// of [lo, i_end).  With ALIGNED the groups end at tile boundaries (the tiles
// of a mixed-precision factor differ in their element type).
template <int R, bool ALIGNED>
__host__ __device__ __forceinline__ int row_groups(int lo, int i_end, int q) {
  if (i_end <= lo) return 0;
  if (!ALIGNED) return (i_end - lo + R - 1) / R;
  const int first = (lo / q + 1) * q;
  if (i_end <= first) return (i_end - lo + R - 1) / R;
  const int rest = i_end - first;
  return (first - lo + R - 1) / R + rest / q * ((q + R - 1) / R) + (rest % q + R - 1) / R;
}
template <int R, bool ALIGNED>
__device__ __forceinline__ void row_group(int t, int lo, int i_end, int q, int& i0, int& nr) {
  int end = i_end;
  i0 = lo + t * R;
  if (ALIGNED) {
    const int first = (lo / q + 1) * q;
    const int g0 = (first - lo + R - 1) / R;
    if (t < g0) {
      end = first < i_end ? first : i_end;
    } else {
      const int gt = (q + R - 1) / R;
      const int tile = (t - g0) / gt;
      i0 = first + tile * q + (t - g0 - tile * gt) * R;
      end = first + (tile + 1) * q < i_end ? first + (tile + 1) * q : i_end;
    }
  }
  nr = end - i0 < R ? end - i0 : R;
}
// First block row of column j's T tasks: row j + 1 belongs to D_{j+1} unless
// j is the last column.
__host__ __device__ __forceinline__ int rows_from(int j, int j1) { return j + 1 < j1 ? j + 2 : j + 1; }

template <int R, bool MIXED, bool RHS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_chol_flow(FlowArgs a) {
  __shared__ __attribute__((aligned(16))) double lds[kDiagLds];
  static_assert(2 * (R + 1) * kPanel <= kDiagLds, "the T tasks' ring");
  __shared__ int sh[2];
  const int tid = threadIdx.x;
  int j = a.j0;
  long base = 0;  // first task of column j
  lds[kId + tid] = tid % 17 == 0 ? 1.0 : 0.0;
  if (RHS && blockIdx.x == 0 && tid == 0) a.clock[0] = wall_clock64();
  for (;;) {
    if (tid == 0) sh[0] = atomicAdd(a.flags + kClaim, 1);
    __syncthreads();
    const long id = sh[0];
    __syncthreads();
    for (; j < a.j1; ++j) {
      const int cnt = 1 + RHS + row_groups<R, MIXED>(rows_from(j, a.j1), a.i_end, a.q);
      if (id < base + cnt) break;
      base += cnt;
    }
    if (j >= a.j1) break;
    const int t = (int)(id - base);
    if (t == 0) {
      task_diag(a, j, lds, sh + 1);
      if (j + 1 == a.j1) {
        for (long e = tid; e < (long)(a.j_pad - a.j1) * 4096; e += 256)
          a.dinv[(long)a.j1 * 4096 + e] = ((e & 4095) % 65 == 0) ? 1.0 : 0.0;
      }
    } else if (RHS && t == 1) {
      task_rhs(a, j, lds, sh + 1);
    } else {
      int i0, nr;
      row_group<R, MIXED>(t - 1 - RHS, rows_from(j, a.j1), a.i_end, a.q, i0, nr);
      if constexpr (MIXED) {
        if (a.v.prec[tile_index(a.v, i0 / a.q, a.k)] != kF64) task_rows<R, float>(a, i0, nr, j, lds, sh + 1);
        else task_rows<R, double>(a, i0, nr, j, lds, sh + 1);
      } else {
        task_rows<R, double>(a, i0, nr, j, lds, sh + 1);
      }
    }
  }
  // The last work-group leaves the counters as it found them.
  if (tid == 0) sh[0] = atomicAdd(a.flags + kExit, 1) == (int)gridDim.x - 1;
  __syncthreads();
  if (!sh[0]) return;
  for (int e = tid; e < a.i_end - a.j0 + RHS; e += 256) a.flags[kRows + 16 * e] = 0;
  if (RHS && tid == 0) a.clock[1] = wall_clock64();
  if (tid == 0) a.flags[kClaim] = a.flags[kExit] = a.flags[kDiag] = 0;
}

template <int R, bool MIXED, bool RHS = false>
void launch_flow(const FlowArgs& a, hipStream_t s) {
  struct Room {
    int cus, slots;
  };
  static const Room room = [] {  // by the first thread that comes here; others wait for it
    int dev = 0, n = 0, occ = 1;
    EXA_HIP(hipGetDevice(&dev));
    EXA_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    EXA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_chol_flow<R, MIXED, RHS>, 256, 0));
    return Room{n, n * (occ > 0 ? occ : 1)};
  }();
  // Small matrices wait for the chain, which is faster without a second
  // work-group on its CU (more LDS than half a CU's keeps it away); larger
  // ones for the sums.  Likelihood, one / two work-groups per CU: n = 2,000
  // 437 / 453 us, 3,200 675 / 755, 4,400 1,134 / 1,156, 5,003 1,514 / 1,428,
  // 6,000 2,270 / 2,000.
  constexpr int kChainBlocks = 70, kMoreLds = 16384;
  const bool alone = a.pool && a.i_end - a.j0 <= kChainBlocks;
  const int most = alone ? room.cus : room.slots;
  long tasks = 0;
  for (int j = a.j0; j < a.j1 && tasks < most; ++j)
    tasks += 1 + RHS + row_groups<R, MIXED>(rows_from(j, a.j1), a.i_end, a.q);
  const long grid = tasks < most ? tasks : most;
  hipLaunchKernelGGL((k_chol_flow<R, MIXED, RHS>), dim3((unsigned)grid), dim3(256), alone ? kMoreLds : 0, s, a);
  EXA_HIP(hipGetLastError());
}

// Before a factorisation: info = 0 and the inverses unset; with a right-hand
// side also z into the first row of its blocks.  The other rows are zero since
// their allocation, or NaN once a factorisation has failed: the rows never mix.
__global__ void __launch_bounds__(256) k_flow_begin(const double* z, long n, double* rhs, double* dinv, long nd,
                                                    int* info) {
  const long c = (long)blockIdx.x * 256 + threadIdx.x;
  if (c == 0) *info = 0;
  // The padding too (nd / 64 columns): the buffer serves matrices of several
  // orders, and a NaN left there would spread over its block as 0 * NaN.
  if (c < nd / kNB) rhs[c * kNB] = c < n ? z[c] : 0.0;
  for (long e = c; e < nd; e += (long)gridDim.x * 256) reinterpret_cast<long long*>(dinv)[e] = kUnset;
}
__global__ void __launch_bounds__(256) k_flow_reset(double* dinv, long nd, int* info) {
  const long c = (long)blockIdx.x * 256 + threadIdx.x;
  if (c == 0) *info = 0;
  for (long e = c; e < nd; e += (long)gridDim.x * 256) reinterpret_cast<long long*>(dinv)[e] = kUnset;
}

// After it: y = L^-1 z into a vector (zeros into its padding, which a solve on
// the tiles may have left as NaN and the transposed solve reads), and per
// work-group the sums of y^2 and of log L_ii over 256 rows, written with info
// and the phases' ticks to host memory.
__global__ void __launch_bounds__(256) k_flow_end(TileView v, const double* rhs, long n, double* y, const int* info,
                                                  const long long* clock, double* host, bool keep) {
  __shared__ double red[2][4];
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  double s = 0.0, d = 0.0;
  if (i < n) {
    const double w = rhs[i * kNB];
    if (!keep || *info == 0) y[i] = w;
    s = w * w;
    const int k = (int)(i / v.ts);
    const long r = i - (long)k * v.ts;
    const double l = tile_f64(v, k, k)[r + r * v.ts];
    if (l > 0.0) d = log(l);
  } else if (i < (long)v.mt * v.ts && !keep) {
    y[i] = 0.0;
  }
  s = wave_sum(s);
  d = wave_sum(d);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = s;
    red[1][threadIdx.x >> 6] = d;
  }
  __syncthreads();
  if (threadIdx.x < 2 && (long)blockIdx.x * 256 < n) {
    const double* r = red[threadIdx.x];
    host[4 + 2 * blockIdx.x + threadIdx.x] = (r[0] + r[1]) + (r[2] + r[3]);
  }
  if (i == 0) {
    host[0] = *info;
    host[1] = (double)(clock[2] - clock[0]);
    host[2] = (double)(clock[1] - clock[2]);
    host[3] = (double)(wall_clock64() - clock[1]);
  }
}

}  // namespace

long chol_flow_flags(int mt, int ts) { return kRows + 16L * (mt * (ts / kNB) + 1); }

void launch_chol_flow(const TileView& v, double* pool, int tile_col, int j0, int j1, int i_end, int j_pad,
                      double* dinv, int* info, int* flags, hipStream_t s, double* rhs, long long* clock) {
  FlowArgs a;
  a.v = v;
  a.pool = pool;
  a.k = tile_col;
  a.q = v.ts / kNB;
  a.j0 = j0;
  a.j1 = j1;
  a.i_end = i_end;
  a.j_pad = j_pad;
  a.dinv = dinv;
  a.info = info;
  a.flags = flags;
  a.rhs = rhs;
  a.clock = clock;
  const int nb = v.mt * a.q;
  if (!v.lower || j0 < 0 || j1 <= j0 || j1 > nb || i_end < j1 || i_end > nb || j_pad > nb)
    throw std::invalid_argument("chol_flow: block range outside the matrix");
  if (rhs && (!pool || !clock)) throw std::invalid_argument("chol_flow: right-hand sides go with the whole matrix and a clock");
  if (!pool && (tile_col < 0 || j0 < tile_col * a.q || j1 > (tile_col + 1) * a.q))
    throw std::invalid_argument("chol_flow: block columns outside the tile column");
  if (rhs) launch_flow<2, false, true>(a, s);
  else if (pool) launch_flow<2, false>(a, s);
  else if (v.prec) launch_flow<3, true>(a, s);
  else launch_flow<3, false>(a, s);
}

void launch_flow_begin(const double* z, long n, double* rhs, double* dinv, long nd, int* info, hipStream_t s) {
  hipLaunchKernelGGL(k_flow_begin, dim3((unsigned)(nd / 2048 + (n + 255) / 256)), dim3(256), 0, s, z, n, rhs, dinv, nd, info);
  EXA_HIP(hipGetLastError());
}
void launch_flow_reset(double* dinv, long nd, int* info, hipStream_t s) {
  hipLaunchKernelGGL(k_flow_reset, dim3((unsigned)(nd / 2048 + 1)), dim3(256), 0, s, dinv, nd, info);
  EXA_HIP(hipGetLastError());
}
long flow_end_doubles(long n) { return 4 + 2 * ((n + 255) / 256); }
void launch_flow_end(const TileView& v, const double* rhs, long n, double* y, const int* info, const long long* clock,
                     double* host, bool keep, hipStream_t s) {
  const long padded = (long)v.mt * v.ts;
  hipLaunchKernelGGL(k_flow_end, dim3((unsigned)((padded + 255) / 256)), dim3(256), 0, s, v, rhs, n, y, info, clock,
                     host, keep);
  EXA_HIP(hipGetLastError());
}

}  // namespace exa
