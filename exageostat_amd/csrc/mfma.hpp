// FP64 MFMA work-group GEMM core for CDNA4 (gfx950).
//
// acc += sign * A * B^T, A: BM x K, B: BN x K, both column-major in global
// memory.  A and B are staged through LDS in BK-deep slices, either with
// register-staged double buffering (gemm_nt_acc: global loads of slice k+1
// are in flight while slice k feeds the matrix cores; FP32 and K-major
// operands) or with direct-to-LDS copies into a ring and software-pipelined
// fragments (gemm_nt_pipe: plain FP64 operands).  Each 64-lane wave owns a WM x WN
// sub-block made of 16x16 fragments of v_mfma_f64_16x16x4f64.
#pragma once

#include "common.hpp"

#include <cstdint>

namespace exa {

typedef double dx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ dx4 mfma_f64(double a, double b, dx4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// v_mfma_f64_16x16x4f64 operand/result layouts (64 lanes):
//   A (16x4): lane l supplies A[l%16][l/16];  B (4x16): B[l/16][l%16];
//   D (16x16): lane l, element v holds D[l/16 + 4*v][l%16]
//   (measured on gfx950 with an in-bounds single-wave probe).
__device__ __forceinline__ int frag_row(int lane, int v) { return (lane >> 4) + 4 * v; }
__device__ __forceinline__ int frag_col(int lane) { return lane & 15; }

template <int BM_, int BN_, int WGM_, int WGN_, int BK_>
struct GemmCfg {
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, BK = BK_;
  static constexpr int NW = WGM * WGN;
  static constexpr int NT = NW * 64;
  static constexpr int WM = BM / WGM, WN = BN / WGN;
  static constexpr int FM = WM / 16, FN = WN / 16;
  static constexpr int PAD = 4;
  static constexpr int LDA = BM + PAD, LDB = BN + PAD;
  static constexpr int A_STAGE = BK * LDA, B_STAGE = BK * LDB;
  static constexpr int LDS_DOUBLES = 2 * (A_STAGE + B_STAGE);
  static constexpr int A_LOADS = BM * BK / 2 / NT;
  static constexpr int B_LOADS = BN * BK / 2 / NT;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be 16-aligned");
  static_assert(A_LOADS * NT * 2 == BM * BK, "A slice must split evenly");
  static_assert(B_LOADS * NT * 2 == BN * BK, "B slice must split evenly");
};

// Loads through an explicit global (address space 1) pointer: the tile
// pointers come from a table, so without the cast the compiler emits flat
// loads whose completion it can only wait for together with LDS traffic.
__device__ __forceinline__ double2 ld_global2(const double* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(1))) const double2 gdouble2;
  return *reinterpret_cast<gdouble2*>(reinterpret_cast<uintptr_t>(p));
#else
  return *reinterpret_cast<const double2*>(p);
#endif
}

__device__ __forceinline__ float2 ld_global_f2(const float* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(1))) const float2 gfloat2;
  return *reinterpret_cast<gfloat2*>(reinterpret_cast<uintptr_t>(p));
#else
  return *reinterpret_cast<const float2*>(p);
#endif
}

// Two consecutive elements of a tile stored as T, loaded raw (Pair<T>) and
// widened to FP64 only when stored to LDS, so the loads of the next slice
// stay in flight while the current one is multiplied.
template <class T>
struct Pair;
template <>
struct Pair<double> {
  using type = double2;
};
template <>
struct Pair<float> {
  using type = float2;
};
__device__ __forceinline__ double2 ld_raw(const double* p) { return ld_global2(p); }
__device__ __forceinline__ float2 ld_raw(const float* p) { return ld_global_f2(p); }
__device__ __forceinline__ double2 widen(double2 v) { return v; }
__device__ __forceinline__ double2 widen(float2 v) { return double2{(double)v.x, (double)v.y}; }

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void glb_void_t;

// Waits until at most n vector-memory operations of this wave are pending
// (expcnt and lgkmcnt left at their maxima).  For the direct-to-LDS copies
// the counter drops when the data is in LDS.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

template <class C>
__device__ __forceinline__ void zero_acc(dx4 (&acc)[C::FM][C::FN]) {
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) acc[i][j] = dx4{0.0, 0.0, 0.0, 0.0};
}

// K must be a multiple of BK; lda/ldb even and A/B 16-byte aligned.
// B_KMAJOR: B is given as K x BN column-major (B(k, c) at B[k + c*ldb])
// instead of BN x K; A_KMAJOR likewise for A (A(r, k) at A[k + r*lda]).
// TA/TB: storage type of A/B (FP32 tiles of the mixed-precision factor are
// widened on load).  Ends with a barrier, so the caller may reuse the LDS.
template <class C, bool B_KMAJOR = false, class TA = double, class TB = double, bool A_KMAJOR = false>
__device__ __forceinline__ void gemm_nt_acc(dx4 (&acc)[C::FM][C::FN], const TA* __restrict__ A, long lda,
                                            const TB* __restrict__ B, long ldb, int K, double* lds,
                                            double sign) {
  if (K <= 0) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  double* As = lds;
  double* Bs = lds + 2 * C::A_STAGE;
  typename Pair<TA>::type ra[C::A_LOADS];
  typename Pair<TB>::type rb[C::B_LOADS];

  auto gload = [&](int k0) {
#pragma unroll
    for (int t = 0; t < C::A_LOADS; ++t) {
      const int e = tid + t * C::NT;
      if (A_KMAJOR) {
        const int r = e / (C::BK / 2);
        const int k2 = e - r * (C::BK / 2);
        ra[t] = ld_raw(A + (long)r * lda + k0 + 2 * k2);
      } else {
        const int c = e / (C::BM / 2);
        const int r2 = e - c * (C::BM / 2);
        ra[t] = ld_raw(A + (long)(k0 + c) * lda + 2 * r2);
      }
    }
#pragma unroll
    for (int t = 0; t < C::B_LOADS; ++t) {
      const int e = tid + t * C::NT;
      if (B_KMAJOR) {
        const int c = e / (C::BK / 2);
        const int k2 = e - c * (C::BK / 2);
        rb[t] = ld_raw(B + (long)c * ldb + k0 + 2 * k2);
      } else {
        const int c = e / (C::BN / 2);
        const int r2 = e - c * (C::BN / 2);
        rb[t] = ld_raw(B + (long)(k0 + c) * ldb + 2 * r2);
      }
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int t = 0; t < C::A_LOADS; ++t) {
      const int e = tid + t * C::NT;
      if (A_KMAJOR) {
        const int r = e / (C::BK / 2);
        const int k2 = e - r * (C::BK / 2);
        const double2 w = widen(ra[t]);
        As[buf * C::A_STAGE + (2 * k2) * C::LDA + r] = w.x;
        As[buf * C::A_STAGE + (2 * k2 + 1) * C::LDA + r] = w.y;
      } else {
        const int c = e / (C::BM / 2);
        const int r2 = e - c * (C::BM / 2);
        *reinterpret_cast<double2*>(As + buf * C::A_STAGE + c * C::LDA + 2 * r2) = widen(ra[t]);
      }
    }
#pragma unroll
    for (int t = 0; t < C::B_LOADS; ++t) {
      const int e = tid + t * C::NT;
      if (B_KMAJOR) {
        const int c = e / (C::BK / 2);
        const int k2 = e - c * (C::BK / 2);
        const double2 w = widen(rb[t]);
        Bs[buf * C::B_STAGE + (2 * k2) * C::LDB + c] = w.x;
        Bs[buf * C::B_STAGE + (2 * k2 + 1) * C::LDB + c] = w.y;
      } else {
        const int c = e / (C::BN / 2);
        const int r2 = e - c * (C::BN / 2);
        *reinterpret_cast<double2*>(Bs + buf * C::B_STAGE + c * C::LDB + 2 * r2) = widen(rb[t]);
      }
    }
  };

  const int nk = K / C::BK;
  gload(0);
  sstore(0);
  __syncthreads();
  for (int kc = 0; kc < nk; ++kc) {
    const int buf = kc & 1;
    if (kc + 1 < nk) gload((kc + 1) * C::BK);
    const double* Ab = As + buf * C::A_STAGE + wm * C::WM + (lane & 15);
    const double* Bb = Bs + buf * C::B_STAGE + wn * C::WN + (lane & 15);
#pragma unroll
    for (int kk = 0; kk < C::BK; kk += 4) {
      const int krow = kk + (lane >> 4);
      double a[C::FM], b[C::FN];
#pragma unroll
      for (int i = 0; i < C::FM; ++i) a[i] = sign * Ab[krow * C::LDA + i * 16];
#pragma unroll
      for (int j = 0; j < C::FN; ++j) b[j] = Bb[krow * C::LDB + j * 16];
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int j = 0; j < C::FN; ++j) acc[i][j] = mfma_f64(a[i], b[j], acc[i][j]);
    }
    // Keep the LDS stores of the prefetched slice after the matrix-core work
    // (otherwise they are hoisted next to the global loads and every slice
    // waits for memory before its MFMAs).
    __builtin_amdgcn_sched_barrier(0);
    if (kc + 1 < nk) sstore(buf ^ 1);
    __syncthreads();
  }
}

// The same product for plain FP64 operands, software-pipelined, with the
// fragments the other way round: acc[i][j] holds the block of rows
// 16 i .. and columns 16 j .. with lane l, element v at row l%16, column
// l/16 + 4 v (v_mfma_f64_16x16x4f64 with B's fragment as its first operand),
// so 16 lanes of an access to a column-major block are 128 contiguous bytes.
// The products and their order of summation are those of gemm_nt_acc.
//
// Bound by the FP64 matrix cores (64 cycles per instruction and SIMD).  What
// keeps them fed, with 15,360 x 15,360 x 1,920 blocks over the whole card
// (the same loop with 192 x 192 blocks, one work-group per CU, unpipelined
// fragments: 62.7 TFLOP/s):
//   * NST-stage LDS ring filled by global_load_lds_dwordx4 (no staging
//     registers): slice kc + NST is requested as soon as slice kc is in
//     registers;
//   * the fragments of the next four k are read from LDS while the current
//     four are multiplied, also across slices, so that no wave waits for LDS
//     after a barrier (192 x 192: 67.7 TFLOP/s);
//   * two 256-thread work-groups per CU, so that one multiplies while the
//     other is at a barrier or writes its block out (96 x 192: 71.5,
//     128 x 128: 68.4, 64 x 64: 60.9 TFLOP/s).
// Stage layout: A as BK columns of BM doubles, then B; odd columns have
// neighbouring groups of 16 rows exchanged (row ^ 16), so the two columns
// that one LDS pass reads lie in different halves of the banks (5.6% of the
// LDS cycles were conflicts without).  A wave-wide copy fills 1,024
// contiguous LDS bytes, lane l taking elements 128 q + 2 l.
// Operands: segment s (0 <= s < nseg) multiplies A_s B_s^T with K columns,
// both from seg(s, A, B) with the leading dimension ld (even; pointers
// 16-byte aligned); K a multiple of BK.
template <class C, int NST>
struct PipeLds {
  static constexpr int A_ST = C::BK * C::BM, B_ST = C::BK * C::BN;  // doubles per stage
  static constexpr int STAGE = A_ST + B_ST;
  static constexpr int DOUBLES = NST * STAGE;
  static constexpr int A_COPIES = A_ST / 128, B_COPIES = B_ST / 128;
  static constexpr int PER_WAVE = (A_COPIES + B_COPIES) / C::NW;
  static_assert(A_ST % 128 == 0 && B_ST % 128 == 0, "stage arrays must be whole 1 KB copies");
  static_assert(PER_WAVE * C::NW == A_COPIES + B_COPIES, "copies must split evenly over the waves");
  static_assert(C::BM % 32 == 0 && C::BN % 32 == 0, "row groups are exchanged in pairs");
  static_assert(NST >= 2 && NST * PER_WAVE < 64, "vmcnt range");
};

// Waits until at most n vector-memory operations and no LDS operation of
// this wave are pending.
template <int N>
__device__ __forceinline__ void wait_vmcnt_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4));
}

template <class C, int NST, class SEG>
__device__ __forceinline__ void gemm_nt_pipe(dx4 (&acc)[C::FM][C::FN], int nseg, const SEG& seg, long ld, int K,
                                             double* lds) {
  using L = PipeLds<C, NST>;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  const int per_seg = K / C::BK;
  const int nk = nseg * per_seg;
  if (nk <= 0) return;
  uint32_t off[L::PER_WAVE];  // byte offset of this lane's element in a slice of its operand
#pragma unroll
  for (int j = 0; j < L::PER_WAVE; ++j) {
    int c = wave * L::PER_WAVE + j;
    const bool is_b = c >= L::A_COPIES;
    if (is_b) c -= L::A_COPIES;
    const int rows = is_b ? C::BN : C::BM;
    const int e = c * 128 + 2 * lane;
    const int kk = e / rows;
    const int r = (e - kk * rows) ^ ((kk & 1) * 16);
    off[j] = (uint32_t)((r + kk * (int)ld) * 8);
  }
  const double *A, *B;
  seg(0, A, B);
  int s_next = 1, left = per_seg;  // next segment, slices left in the current one
  auto issue = [&](int buf) {
    if (left == 0) {
      seg(s_next++, A, B);
      left = per_seg;
    }
#pragma unroll
    for (int j = 0; j < L::PER_WAVE; ++j) {
      int c = wave * L::PER_WAVE + j;
      const bool is_b = c >= L::A_COPIES;
      if (is_b) c -= L::A_COPIES;
      const char* src = reinterpret_cast<const char*>(is_b ? B : A) + off[j];
      double* dst = lds + buf * L::STAGE + (is_b ? L::A_ST : 0) + c * 128;
      __builtin_amdgcn_global_load_lds((glb_void_t*)(uintptr_t)src, (lds_void_t*)dst, 16, 0, 0);
    }
    A += (long)C::BK * ld;
    B += (long)C::BK * ld;
    --left;
  };
  const int flip = ((lane >> 4) & 1) * 16;
  const int a0 = wm * C::WM, b0 = wn * C::WN;
  const int ao = (lane & 15) + (lane >> 4) * C::BM;
  const int bo = (lane & 15) + (lane >> 4) * C::BN + L::A_ST;
  double a[2][C::FM], b[2][C::FN];
  auto frag = [&](int set, int buf, int kk) {
    const double* Ab = lds + buf * L::STAGE + ao + kk * 4 * C::BM;
    const double* Bb = lds + buf * L::STAGE + bo + kk * 4 * C::BN;
#pragma unroll
    for (int i = 0; i < C::FM; ++i) a[set][i] = Ab[(a0 + i * 16) ^ flip];
#pragma unroll
    for (int j = 0; j < C::FN; ++j) b[set][j] = Bb[(b0 + j * 16) ^ flip];
  };
  constexpr int NK = C::BK / 4;
  static_assert(NK % 2 == 0, "the two fragment sets alternate over a slice");
  // The ring may still be read by the previous block's last steps.
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int st = 0; st < NST; ++st)
    if (st < nk) issue(st);
  if (nk >= NST) wait_vmcnt<(NST - 1) * L::PER_WAVE>();
  else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  frag(0, 0, 0);
  int buf = 0;
#pragma unroll 1
  for (int kc = 0; kc < nk; ++kc) {
    const int nbuf = buf == NST - 1 ? 0 : buf + 1;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const int cur = kk & 1, nxt = cur ^ 1;
      if (kk + 1 < NK) {
        frag(nxt, buf, kk + 1);
      } else if (kc + 1 < nk) {
        // Slice kc + 1 has landed, and every wave holds its last fragments
        // of slice kc, whose buffer can be filled again.
        __builtin_amdgcn_sched_barrier(0);
        if (kc + NST - 1 < nk) wait_vmcnt_lgkm0<(NST - 2) * L::PER_WAVE>();
        else wait_vmcnt_lgkm0<0>();
        __builtin_amdgcn_s_barrier();
        if (kc + NST < nk) issue(buf);
        frag(nxt, nbuf, 0);
      }
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int j = 0; j < C::FN; ++j) acc[i][j] = mfma_f64(b[cur][j], a[cur][i], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    buf = nbuf;
  }
}

// Base pointer of this lane's elements of a block in gemm_nt_pipe's layout.
template <class C>
__device__ __forceinline__ auto pipe_base(double* Cp, long ldc) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  typedef __attribute__((address_space(1))) double gD;
  return (gD*)(uintptr_t)(Cp + wm * C::WM + (lane & 15) + (long)(wn * C::WN + (lane >> 4)) * ldc);
}

// C -= acc, one fragment column at a time with all its reads before its
// writes.
template <class C>
__device__ __forceinline__ void pipe_sub(const dx4 (&acc)[C::FM][C::FN], double* Cp, long ldc) {
  auto* G = pipe_base<C>(Cp, ldc);
#pragma unroll
  for (int j = 0; j < C::FN; ++j) {
    double cv[4][C::FM];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int i = 0; i < C::FM; ++i) cv[v][i] = G[i * 16 + (long)(j * 16 + 4 * v) * ldc];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int i = 0; i < C::FM; ++i) G[i * 16 + (long)(j * 16 + 4 * v) * ldc] = cv[v][i] - acc[i][j][v];
  }
}

// C = acc.
template <class C>
__device__ __forceinline__ void pipe_put(const dx4 (&acc)[C::FM][C::FN], double* Cp, long ldc) {
  auto* G = pipe_base<C>(Cp, ldc);
#pragma unroll
  for (int j = 0; j < C::FN; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int i = 0; i < C::FM; ++i) G[i * 16 + (long)(j * 16 + 4 * v) * ldc] = acc[i][j][v];
}

// C = -acc.
template <class C>
__device__ __forceinline__ void pipe_put_neg(const dx4 (&acc)[C::FM][C::FN], double* Cp, long ldc) {
  auto* G = pipe_base<C>(Cp, ldc);
#pragma unroll
  for (int j = 0; j < C::FN; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int i = 0; i < C::FM; ++i) G[i * 16 + (long)(j * 16 + 4 * v) * ldc] = -acc[i][j][v];
}

// Cp[c + r*ldc] = -acc(r, c): the block stored transposed.
template <class C>
__device__ __forceinline__ void pipe_put_neg_t(const dx4 (&acc)[C::FM][C::FN], double* Cp, long ldc) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  typedef __attribute__((address_space(1))) double gD;
  gD* G = (gD*)(uintptr_t)(Cp + wn * C::WN + (lane >> 4) + (long)(wm * C::WM + (lane & 15)) * ldc);
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) G[j * 16 + 4 * v + (long)(i * 16) * ldc] = -acc[i][j][v];
}

// C[r + c*ldc] = beta*C + acc for the block owned by this work-group.
template <class C, class T = double>
__device__ __forceinline__ void acc_update(dx4 (&acc)[C::FM][C::FN], T* Cp, long ldc, double beta) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  // Global-address-space accesses, one fragment row at a time with all its
  // reads issued before its writes: with generic read-modify-writes the
  // compiler must assume that a store may alias the next load and
  // serialises the block's memory traffic.
  typedef __attribute__((address_space(1))) T gT;
  gT* G = (gT*)(uintptr_t)Cp;
#pragma unroll
  for (int i = 0; i < C::FM; ++i) {
    if (beta != 0.0) {
      T cv[C::FN][4];
#pragma unroll
      for (int j = 0; j < C::FN; ++j) {
        const int c = wn * C::WN + j * 16 + frag_col(lane);
#pragma unroll
        for (int v = 0; v < 4; ++v) cv[j][v] = G[wm * C::WM + i * 16 + frag_row(lane, v) + (long)c * ldc];
      }
#pragma unroll
      for (int j = 0; j < C::FN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] = beta * (double)cv[j][v] + acc[i][j][v];
    }
#pragma unroll
    for (int j = 0; j < C::FN; ++j) {
      const int c = wn * C::WN + j * 16 + frag_col(lane);
#pragma unroll
      for (int v = 0; v < 4; ++v) G[wm * C::WM + i * 16 + frag_row(lane, v) + (long)c * ldc] = (T)acc[i][j][v];
    }
  }
}

// ---------------------------------------------------- FP32 matrix cores --
// v_mfma_f32_16x16x4f32: operands as for the FP64 instruction (lane l
// supplies A[l%16][l/16] and B[l/16][l%16]); result: lane l, element v holds
// D[4*(l/16)+v][l%16].
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <class C>
__device__ __forceinline__ void zero_acc32(f32x4 (&acc)[C::FM][C::FN]) {
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// acc += sign * A * B^T with FP64 operands rounded to FP32 when staged into
// LDS (the register-staged double buffering of gemm_nt_acc, plain operand
// layout) and FP32 matrix cores at twice the FP64 rate, FP32 accumulation.
// lds: C::LDS_DOUBLES doubles, used as twice as many floats' worth of half.
template <class C>
__device__ __forceinline__ void gemm_nt_acc32(f32x4 (&acc)[C::FM][C::FN], const double* __restrict__ A, long lda,
                                              const double* __restrict__ B, long ldb, int K, float* lds,
                                              float sign) {
  if (K <= 0) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  float* As = lds;
  float* Bs = lds + 2 * C::A_STAGE;
  double2 ra[C::A_LOADS];
  double2 rb[C::B_LOADS];
  auto gload = [&](int k0) {
#pragma unroll
    for (int t = 0; t < C::A_LOADS; ++t) {
      const int e = tid + t * C::NT;
      const int c = e / (C::BM / 2);
      const int r2 = e - c * (C::BM / 2);
      ra[t] = ld_global2(A + (long)(k0 + c) * lda + 2 * r2);
    }
#pragma unroll
    for (int t = 0; t < C::B_LOADS; ++t) {
      const int e = tid + t * C::NT;
      const int c = e / (C::BN / 2);
      const int r2 = e - c * (C::BN / 2);
      rb[t] = ld_global2(B + (long)(k0 + c) * ldb + 2 * r2);
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int t = 0; t < C::A_LOADS; ++t) {
      const int e = tid + t * C::NT;
      const int c = e / (C::BM / 2);
      const int r2 = e - c * (C::BM / 2);
      *reinterpret_cast<float2*>(As + buf * C::A_STAGE + c * C::LDA + 2 * r2) =
          float2{(float)ra[t].x, (float)ra[t].y};
    }
#pragma unroll
    for (int t = 0; t < C::B_LOADS; ++t) {
      const int e = tid + t * C::NT;
      const int c = e / (C::BN / 2);
      const int r2 = e - c * (C::BN / 2);
      *reinterpret_cast<float2*>(Bs + buf * C::B_STAGE + c * C::LDB + 2 * r2) =
          float2{(float)rb[t].x, (float)rb[t].y};
    }
  };
  const int nk = K / C::BK;
  gload(0);
  sstore(0);
  __syncthreads();
  for (int kc = 0; kc < nk; ++kc) {
    const int buf = kc & 1;
    if (kc + 1 < nk) gload((kc + 1) * C::BK);
    const float* Ab = As + buf * C::A_STAGE + wm * C::WM + (lane & 15);
    const float* Bb = Bs + buf * C::B_STAGE + wn * C::WN + (lane & 15);
#pragma unroll
    for (int kk = 0; kk < C::BK; kk += 4) {
      const int krow = kk + (lane >> 4);
      float a[C::FM], b[C::FN];
#pragma unroll
      for (int i = 0; i < C::FM; ++i) a[i] = sign * Ab[krow * C::LDA + i * 16];
#pragma unroll
      for (int j = 0; j < C::FN; ++j) b[j] = Bb[krow * C::LDB + j * 16];
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int j = 0; j < C::FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (kc + 1 < nk) sstore(buf ^ 1);
    __syncthreads();
  }
}

// Cp[r + c*ldc] = acc(r, c) as FP64 (the FP32 result layout).
template <class C>
__device__ __forceinline__ void acc32_store(const f32x4 (&acc)[C::FM][C::FN], double* Cp, long ldc) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  typedef __attribute__((address_space(1))) double gD;
  gD* G = (gD*)(uintptr_t)(Cp + wm * C::WM + 4 * (lane >> 4) + (long)(wn * C::WN + (lane & 15)) * ldc);
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) G[i * 16 + v + (long)j * 16 * ldc] = (double)acc[i][j][v];
}

// Cp[c + r*ldc] = acc(r, c) as FP64: the block stored transposed.
template <class C>
__device__ __forceinline__ void acc32_store_t(const f32x4 (&acc)[C::FM][C::FN], double* Cp, long ldc) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  typedef __attribute__((address_space(1))) double gD;
  gD* G = (gD*)(uintptr_t)(Cp + wn * C::WN + (lane & 15) + (long)(wm * C::WM + 4 * (lane >> 4)) * ldc);
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const long ro = (long)(i * 16 + v) * ldc;
#pragma unroll
      for (int j = 0; j < C::FN; ++j) G[ro + j * 16] = (double)acc[i][j][v];
    }
}

}  // namespace exa
