// Lower-precision MFMA work-group GEMM core for the mixed-precision tile
// Cholesky on CDNA4 (gfx950): BF16 operands (single or split in two BF16
// terms) with FP32 accumulation (v_mfma_f32_16x16x32_bf16).
//
// It computes acc += A * B^T for a BM x BN block from panel tiles that were
// converted once per step into BF16 parts (k_split_panel), copied into a
// ring in LDS with direct-to-LDS loads, and read from there one step ahead.
// Result layout (measured on gfx950 with an in-bounds single-wave probe):
// lane l, element v holds D[4*(l/16)+v][l%16]; operand layout: lane l holds
// A[l%16][8*(l/16)+e] and B^T[l%16][8*(l/16)+e], e = 0..7.
#pragma once

#include "common.hpp"
#include "mfma.hpp"

#include <type_traits>

namespace exa {

typedef float fx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ int frag_row_lp(int lane, int v) { return 4 * (lane >> 4) + v; }

template <int BM_, int BN_, int WGM_, int WGN_, int BK_>
struct LpCfg {
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, BK = BK_;
  static constexpr int NW = WGM * WGN;
  static constexpr int NT = NW * 64;
  static constexpr int WM = BM / WGM, WN = BN / WGN;
  static constexpr int FM = WM / 16, FN = WN / 16;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be 16-aligned");
};

template <class C>
__device__ __forceinline__ void zero_acc_lp(fx4 (&acc)[C::FM][C::FN]) {
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) acc[i][j] = fx4{0.f, 0.f, 0.f, 0.f};
}

// C[r + c*ldc] += sign * acc (C stored as T); acc is overwritten.  Every
// read of C precedes the first write, through global-address-space
// pointers, so the block's reads are issued together instead of one
// read-modify-write at a time.
template <class C, class T>
__device__ __forceinline__ void acc_add_lp(fx4 (&acc)[C::FM][C::FN], T* Cp, long ldc, float sign = 1.f) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  typedef __attribute__((address_space(1))) T gT;
  gT* G = (gT*)(uintptr_t)Cp;
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) {
      const int c = wn * C::WN + j * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = wm * C::WM + i * 16 + frag_row_lp(lane, v);
        acc[i][j][v] = (float)G[r + (long)c * ldc] + sign * acc[i][j][v];
      }
    }
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) {
      const int c = wn * C::WN + j * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = wm * C::WM + i * 16 + frag_row_lp(lane, v);
        G[r + (long)c * ldc] = (T)acc[i][j][v];
      }
    }
}

// ------------------------------------------------------- split BF16 --
// The BF16 update classes multiply BF16 operands on the matrix cores
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation).  NSPLIT = 1: operands
// rounded to BF16.  NSPLIT = 3 or 4: each operand is split as x = hi + lo
// (hi = bf16(x), lo = bf16(x - hi), about 16 significant bits together) and
// the product is hi*hi + hi*lo + lo*hi (+ lo*lo for NSPLIT = 4); products of
// BF16 values are exact in FP32.  The lo*lo term is small (2^-16 relative)
// but not random: rows of neighbouring locations have strongly correlated
// remainders, so dropping it biases A*B^T, and through the Schur complements
// the log-determinant, in one direction.  NSPLIT = 4 runs at a quarter of
// the BF16 rate, several times the FP32 MFMA rate.

typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 b2v __attribute__((ext_vector_type(2)));

// Two FP32 values rounded to BF16 (hardware round-to-nearest-even, one
// packed conversion) and, for NSPLIT >= 3, their BF16 remainders.
template <int NSPLIT>
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& hi, uint32_t& lo) {
  const f2v v = {a, b};
  const b2v h = __builtin_convertvector(v, b2v);
  hi = __builtin_bit_cast(uint32_t, h);
  if (NSPLIT >= 3) {
    const f2v back = __builtin_convertvector(h, f2v);
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(v - back, b2v));
  }
}

// ------------------------------------------- direct-to-LDS operand loads --
// Panel tiles are converted once per step into BF16 hi (and lo) parts (see
// k_split_panel), laid out per tile as [k-group g][row r][8 k values]
// (g = column / 8): one 16-byte load is eight k values of one row, and
// consecutive rows are consecutive in memory.  The lo parts of a tile follow
// its hi parts.
//
// The product copies the operands with
// global_load_lds_dwordx4 (each wave-wide instruction writes 64 lanes x 16
// bytes contiguously into LDS, no registers involved) into a ring of 32-deep
// slices.  The LDS layout of a stage is the panel's own [k-group][row][8]:
// array a (A hi, B hi, A lo, B lo) holds 4 groups of its rows.  A
// 16-lane quarter of a fragment read covers 16 consecutive rows of one
// group, 256 contiguous bytes, so neither the copies nor the reads conflict
// on LDS banks.
template <class C, int NSPLIT>
struct Bf16dLds {
  static constexpr int G = C::BK / 8;
  static constexpr int NARR = NSPLIT >= 3 ? 2 : 1;
  static constexpr int A_ARR = G * C::BM * 8;  // halves
  static constexpr int B_ARR = G * C::BN * 8;
  static constexpr int STAGE = NARR * (A_ARR + B_ARR);
  static constexpr int NSTAGE = NSPLIT >= 3 ? 3 : 6;
  static constexpr int HALVES = NSTAGE * STAGE;
  static constexpr int CHUNKS = NARR * G * (C::BM + C::BN) / 64;  // wave-wide copies per stage
  static constexpr int PER_WAVE = CHUNKS / C::NW;
  static_assert(C::BK == 32, "one slice is one step of the matrix cores");
  static_assert(C::BM % 64 == 0 && C::BN % 64 == 0, "rows must be whole 64-row chunks");
  static_assert(CHUNKS % C::NW == 0, "copies must split evenly over the waves");
};

// acc += A * B^T (A and B rows from the split panels, so the caller
// subtracts the result), for K a multiple of 64.
//
// What bounds it is the LDS as much as the matrix cores (192 x 192 blocks, a
// slice of the three products: 196 KB through the LDS against 1,728 cycles of
// MFMA per SIMD), so the two have to run at the same time.  Fragments are
// read one column group of B ahead of their use, the rows of A for the next
// slice beside the column groups of the current one, and copies, reads and
// adds stand between the MFMAs, each of which leaves 12 of its 16 cycles to
// other instructions.  One barrier per slice: there every wave's copies of
// the next slice have landed (they are then read), and every wave is past
// the previous slice, whose buffer receives new copies.
// Measured on 224 CUs, 192 x 192 x 960, three products: 39.6 us a block (1.20
// PFLOP/s; 44.7 with the reads of a slice before its MFMAs), 50.2 with the
// update of C from HBM (61); one product 18.0 us (18.7).
template <class C, int NSPLIT>
__device__ __forceinline__ void gemm_nt_bf16d(fx4 (&acc)[C::FM][C::FN], const uint16_t* __restrict__ Ah,
                                                  const uint16_t* __restrict__ Bh, long lo_off, long gs, int K,
                                                  uint16_t* lds) {
  using L = Bf16dLds<C, NSPLIT>;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / C::WGN;
  const int wn = wave - wm * C::WGN;
  // The copy decomposition is uniform per wave: keep it in scalar registers.
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  const unsigned lane16 = lane * 16;
  // copy j of this wave: chunk c = wave * PER_WAVE + j of array (hi/lo,
  // A/B), k-group g, 64-row block rc; lo parts sit lo_off halves after hi.
  auto issue = [&](int kc, int buf, int j) {
    constexpr int per_a = L::G * (C::BM / 64), per_b = L::G * (C::BN / 64);
    int c = wave_s * L::PER_WAVE + j;
    const int pair = c / (per_a + per_b);  // 0: hi, 1: lo
    c -= pair * (per_a + per_b);
    const bool is_b = c >= per_a;
    if (is_b) c -= per_a;
    const int rows = is_b ? C::BN : C::BM;
    const int g = c / (rows / 64);
    const int rc = c - g * (rows / 64);
    const uint16_t* base = is_b ? Bh : Ah;
    const long goff = pair * lo_off + ((long)(kc * L::G + g) * gs + rc * 64) * 8;
    const int loff = buf * L::STAGE + pair * (L::A_ARR + L::B_ARR) + (is_b ? L::A_ARR : 0) + (g * rows + rc * 64) * 8;
    typedef __attribute__((address_space(1))) const char gchar;
    gchar* src = (gchar*)(uintptr_t)(base + goff);  // uniform: one lane offset serves all copies
    __builtin_amdgcn_global_load_lds((glb_void_t*)(src + lane16), (lds_void_t*)(lds + loff), 16, 0, 0);
  };
  constexpr bool SPLIT = NSPLIT >= 3;
  constexpr int S = L::NSTAGE;
  const int nk = K / C::BK;
  const int row = (lane >> 4), r16 = lane & 15;
  const int ao = (row * C::BM + wm * C::WM + r16) * 8, bo = L::A_ARR + (row * C::BN + wn * C::WN + r16) * 8;
  constexpr int LO = L::A_ARR + L::B_ARR;
  bf16x8 ah[2][C::FM], al[SPLIT ? C::FM : 1], bh[2], bl[2];
  auto read_hi = [&](int set, const uint16_t* st, int i) {
    ah[set][i] = *reinterpret_cast<const bf16x8*>(st + ao + i * 128);
  };
  auto read_lo = [&](const uint16_t* st, int i) {
    if constexpr (SPLIT) al[i] = *reinterpret_cast<const bf16x8*>(st + LO + ao + i * 128);
  };
  auto read_b = [&](int set, const uint16_t* st, int j) {
    bh[set] = *reinterpret_cast<const bf16x8*>(st + bo + j * 128);
    if (SPLIT) bl[set] = *reinterpret_cast<const bf16x8*>(st + LO + bo + j * 128);
  };
  // The ring may still be read by the previous block's last steps.
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int st = 0; st < S - 1; ++st)
#pragma unroll
    for (int j = 0; j < L::PER_WAVE; ++j) issue(st < nk ? st : nk - 1, st, j);
  wait_vmcnt<(S - 2) * L::PER_WAVE>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < C::FM; ++i) {
    read_hi(0, lds, i);
    read_lo(lds, i);
  }
  read_b(0, lds, 0);
  int buf = 0;
  constexpr int NP = NSPLIT;                   // products, smallest terms first
  constexpr int SLOTS = NP * C::FM;            // MFMAs per column group
  // A group's MFMAs go in two halves of its row fragments, so that one half's
  // sums are added, one or two values per MFMA, during the other's products.
  constexpr int H = C::FM / 2;
  static_assert(C::FM % 2 == 0, "two halves");
  // Each 32-deep chunk is summed by its own MFMA chain from zero (smallest
  // terms first) and added to the running sum with one round-to-nearest FP32
  // add: the MFMA's internal accumulation is not correctly rounded (about 1
  // ulp of error per instruction, measured on gfx950), and chaining all
  // 3 K / 32 instructions into one accumulator lets that error build up at
  // the running sum's magnitude.
  fx4 t[SPLIT ? C::FM : 1];
#pragma unroll
  for (int i = 0; i < (SPLIT ? C::FM : 1); ++i) t[i] = fx4{0.f, 0.f, 0.f, 0.f};
  auto slice = [&](auto par, int kc) {
    constexpr int P = decltype(par)::value;  // the slice's fragment set of A
    constexpr int FN = C::FN;
    const int nbuf = buf == S - 1 ? 0 : buf + 1;
    const uint16_t* st = lds + buf * L::STAGE;
    const uint16_t* sn = lds + nbuf * L::STAGE;
    const int kn = kc + S - 1 < nk ? kc + S - 1 : nk - 1;  // (past the end: a copy that nothing reads)
    const int bn = buf == 0 ? S - 1 : buf - 1;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int cur = (P * FN + j) & 1;  // B's sets alternate over all column groups
      const int jp = (j + FN - 1) % FN;
      if (j == 0) {
        wait_vmcnt<(S - 3) * L::PER_WAVE>();
        __builtin_amdgcn_s_barrier();
      }
#pragma unroll
      for (int sl = 0; sl < SLOTS; ++sl) {
        const int h = sl / (NP * H), r = sl % (NP * H);
        const int p = NP - 1 - r / H, i = h * H + r % H;  // 3: lo lo, 2: lo hi, 1: hi lo, 0: hi hi
        if constexpr (SPLIT) {
          const bf16x8 x = p >= 2 ? al[i] : ah[P][i], y = p == 3 || p == 1 ? bl[cur] : bh[cur];
          if (p == NP - 1) {
            t[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, fx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          } else {
            t[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, t[i], 0, 0, 0);
          }
        } else {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[P][i], bh[cur], acc[i][j], 0, 0, 0);
        }
        if constexpr (SPLIT) {
#pragma unroll
          for (int e = 4 * r / NP; e < 4 * (r + 1) / NP; ++e) {
            const int ie = (1 - h) * H + e / 4;
            acc[ie][h ? j : jp][e % 4] += t[ie][e % 4];
          }
        }
        // B of the next group; the high parts of the next slice's A in all
        // groups but the last; its low parts in the last one, each over the
        // current one right after its last use (after the last slice: what is
        // there, unused).  Not before a group's first MFMA: the wait for a
        // fragment is a wait for all LDS reads here, since the compiler takes
        // the direct-to-LDS copies for unordered ones.
        if (sl == 1) read_b(cur ^ 1, j + 1 < FN ? st : sn, j + 1 < FN ? j + 1 : 0);
        if (j < FN - 1) {
          const int i0 = j * C::FM / (FN - 1), i1 = (j + 1) * C::FM / (FN - 1);
#pragma unroll
          for (int ia = i0; ia < i1; ++ia) {
            const int at = 3 + (ia - i0) * (SLOTS - 4) / (i1 - i0);
            if ((at < SLOTS ? at : SLOTS - 1) == sl) read_hi(P ^ 1, sn, ia);
          }
        }
        if (SPLIT && j == FN - 1 && r > (NP - 3) * H && r <= (NP - 2) * H) read_lo(sn, h * H + r - (NP - 3) * H - 1);
        if (j == 0) {
#pragma unroll
          for (int c = 0; c < L::PER_WAVE; ++c)
            if (c * SLOTS / L::PER_WAVE == sl) issue(kn, bn, c);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    buf = nbuf;
  };
#pragma unroll 1
  for (int kc = 0; kc < nk; kc += 2) {
    slice(std::integral_constant<int, 0>{}, kc);
    slice(std::integral_constant<int, 1>{}, kc + 1);
  }
  if constexpr (SPLIT) {
#pragma unroll
    for (int i = H; i < C::FM; ++i) acc[i][C::FN - 1] += t[i];
  }
  wait_vmcnt<0>();
}

}  // namespace exa
