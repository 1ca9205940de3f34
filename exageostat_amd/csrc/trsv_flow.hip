// Triangular solve with the tile factor, z <- L^-1 z or L^-T z, in one
// launch.
//
// Replaces, from EXAGEOSTAT_dmle_Tile (exageostat_exact/src/compute/
// MLE_dexact.c:381-399), CHAMELEON_dtrsm_Tile(Left, Lower, NoTrans, NonUnit)
// on Z, and from EXAGEOSTAT_dmle_Predict_Tile (:812-820) the two triangular
// solves of dposv.
//
// Left-looking over the tiles t = 0, 1, .. of the solve's order (tile t, or
// mt - 1 - t for the transposed solve), with X_t = L_tt^-1:
//   U_t: w_t = z_t - sum_{u < t} L_tu y_u      (transposed: L_ut^T)
//   B_t: y_t = X_t w_t                         (transposed: X_t^T)
// What bounds it is the chain of U_t's last product and B_t, tile after
// tile, and beside it the one pass over L.  Every 64 x 64 block of a tile is
// small against that chain, so a tile's q x q blocks (q = ts / 64) are dealt
// out in strips of up to four: a work-group owns one strip position (a
// block of results and a part of up to four operand blocks), holds the
// strip of the tile to come in registers while it waits for that tile's
// operand, and leaves a partial result; the readers add the at most four
// partials in a fixed order, so the result does not depend on the schedule.
// Four blocks are what 256 threads hold with two work-groups per CU (128
// registers a thread).
//
// Tasks are claimed from one counter in an order in which each depends on
// earlier ones only, and a work-group finishes its task before it claims
// another, so the launch drains whatever share of it is resident.
//
// Measured against two launches per tile (a product with X_t whose last
// work-group adds the partials, an update of the rest of z), per solve:
// n = 900, tiles of 64: 57 us against 174; n = 6,000, tiles of 384: 98 and 90 us
// (forward, transposed) against 270; n = 20,000, tiles of 960: 0.40 ms
// against 0.95; n = 30,720, mixed tiles of 960: 0.51 and 0.48 ms against 1.45,
// where reading L takes 0.4.  With release and acquire at agent scope in
// place of flag_put and load_through the last is 0.67 ms: each of the 3,800
// tasks then writes back an L2.
#include "flow.hpp"
#include "kernels.hpp"

namespace exa {

namespace {

constexpr int kClaim = 0, kExit = 16, kTile = 32;  // flags: 64 for y_t, 64 for w_t, per t

struct TrsvArgs {
  TileView v;
  const double* xinv;  // mt inverses of the diagonal tiles
  double* z;
  double* part;  // per t: parts x ts partials of y_t, then of L_tu y_u
  int* flags;
  int q, parts, per;  // blocks per tile row, parts, blocks per part
};

// sum over the wave's lanes of s[j], j < 16: the lanes 4 j .. 4 j + 3 get
// column j's.
__device__ __forceinline__ double wave_sum16(double (&s)[16], int lane) {
#pragma unroll
  for (int h = 8; h > 0; h >>= 1) {
    const bool up = lane & (4 * h);
#pragma unroll
    for (int j = 0; j < h; ++j) {
      const double lo = s[j], hi = s[j + h];
      s[j] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, 4 * h, 64);
    }
  }
  double x = s[0];
  x += __shfl_xor(x, 2, 64);
  x += __shfl_xor(x, 1, 64);
  return x;
}

// One wave's 16 columns of PER 64 x 64 blocks, step elements apart, the
// lane's row of each; p is the same in all lanes.  A strip of fewer blocks
// reads its last one again (times zeros).  Single-precision values stay as
// they are in the low words until they are used, so that both kinds of tiles
// share the registers.
template <int PER, class T>
__device__ __forceinline__ void load_blocks(const T* p, int ts, int step, int nb, int lane, double (&a)[PER][16]) {
  typedef __attribute__((address_space(1))) const T gT;
#pragma unroll
  for (int b = 0; b < PER; ++b) {
    gT* g = (gT*)(uintptr_t)(p + (long)(b < nb ? b : nb - 1) * step);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const T x = g[(unsigned)lane];
      if constexpr (sizeof(T) == 4) a[b][j] = __longlong_as_double((long long)(unsigned long long)__float_as_uint(x));
      else a[b][j] = x;
      g += ts;
    }
  }
}

template <class T>
__device__ __forceinline__ double held(double a) {
  if constexpr (sizeof(T) == 4) return (double)__uint_as_float((unsigned)__double_as_longlong(a));
  else return a;
}

// acc += blocks (held as T) times the operand blocks at ys.
template <class T, bool TRANS, int PER>
__device__ __forceinline__ void times_blocks(const double (&a)[PER][16], const double* ys, int lane, int wave,
                                             double (&acc)[16]) {
#pragma unroll
  for (int b = 0; b < PER; ++b) {
    if constexpr (TRANS) {
      const double y = ys[b * kNB + lane];
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[j] += held<T>(a[b][j]) * y;
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[j & 3] += held<T>(a[b][j]) * ys[b * kNB + wave * 16 + j];
    }
  }
}

// p[c ts] over the partials c in [first, last), at most four.
__device__ __forceinline__ double sum_parts(const double* p, long ts, int first, int last) {
  double v[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    v[c] = 0.0;
    if (c >= first && c < last) v[c] = load_through(p + c * ts);
  }
  return (v[0] + v[1]) + (v[2] + v[3]);
}

// Waits until every flag f[lane] whose lane is wanted is set.  ahead: how many
// steps of the chain the caller's next use is away; those that are not next
// poll less often, since all polls of a tile's flags meet in one memory
// channel (n = 6,000: 112 us a solve, 236 with every work-group polling at
// full rate).
__device__ __forceinline__ void wait_flags(const int* f, bool wanted, int ahead) {
  if (threadIdx.x < 64) {
    while (!__all(!wanted || flag_get(f + threadIdx.x))) {
      if (ahead > 2) __builtin_amdgcn_s_sleep(64);
      else if (ahead > 0) __builtin_amdgcn_s_sleep(16);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
  __syncthreads();
}

// The work-group's sums: thread i < 64 returns result i of the block.
template <bool TRANS>
__device__ __forceinline__ double block_sum(double (&acc)[16], double* red, int lane, int wave) {
  if constexpr (TRANS) {
    const double x = wave_sum16(acc, lane);
    if ((lane & 3) == 0) red[wave * 16 + (lane >> 2)] = x;
    __syncthreads();
    return red[lane];
  } else {
    red[wave * 64 + lane] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    __syncthreads();
    return (red[lane] + red[64 + lane]) + (red[128 + lane] + red[192 + lane]);
  }
}

template <bool TRANS, bool MIXED, int PER>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_trsv_flow(TrsvArgs a) {
  constexpr bool ONE = PER == 1;  // U_t and B_t in one task
  __shared__ double ys[PER * kNB], red[256];
  __shared__ int sh;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mt = a.v.mt, q = a.q, qc = q * a.parts;
  const long ts = a.v.ts;
  const int vec = a.parts * a.v.ts;  // partials of one vector of tile t
  const int tasks = ONE ? mt : qc * (2 * mt - 1) + mt;
  auto tile_of = [&](int t) { return TRANS ? mt - 1 - t : t; };
  // partials [first, last) of y's block b
  auto y_first = [&](int b) { return TRANS ? b / a.per : 0; };
  auto y_last = [&](int b) { return TRANS ? a.parts : b / a.per + 1; };
  auto y_value = [&](int t, int i) {
    const int b = i / kNB;
    return sum_parts(a.part + (long)2 * t * vec + i, ts, y_first(b), y_last(b));
  };
  for (;;) {
    if (tid == 0) sh = atomicAdd(a.flags + kClaim, 1);
    __syncthreads();
    const int id = sh;
    __syncthreads();
    if (id >= tasks) break;
    int t, r;
    bool upd, fin = false;
    if constexpr (ONE) {
      t = id;
      r = 0;
      upd = true;
    } else {
      t = (id + qc) / (2 * qc);
      r = id + qc - t * 2 * qc;
      upd = r < qc;
      if (!upd) r -= qc;
      fin = t >= mt;
      if (fin) t = id - qc * (2 * mt - 1);
    }
    const int m = tile_of(t);
    if (fin) {  // the sums of y_t's partials, after every B_t has read z_t
      wait_flags(a.flags + kTile + t * 128, lane < qc && lane % a.parts >= y_first(lane / a.parts) &&
                                               lane % a.parts < y_last(lane / a.parts),
                 3);
      for (int i = tid; i < ts; i += 256) a.z[m * ts + i] = y_value(t, i);
      continue;
    }
    const int own = r / a.parts, c = r - own * a.parts;  // block of results, part of the operand
    int b0 = c * a.per;
    int nb = q - b0 < a.per ? q - b0 : a.per;
    // the wave's first element of block b0 of a strip
    long off0 = TRANS ? (long)b0 * kNB + (own * kNB + wave * 16) * ts : own * kNB + (b0 * kNB + wave * 16) * ts;
    const int step = TRANS ? kNB : kNB * a.v.ts;
    double s[PER][16];
    double acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.0;
    double w = 0.0;
    if (upd) {
      bool f32 = false;
      auto fetch = [&](int u) {
        const long ti = TRANS ? tile_index(a.v, tile_of(u), m) : tile_index(a.v, m, u);
        const void* p = a.v.ptr[ti];
        if constexpr (MIXED) {
          f32 = a.v.prec[ti] != kF64;
          if (f32) {
            load_blocks(static_cast<const float*>(p) + off0, a.v.ts, step, nb, lane, s);
            return;
          }
        }
        load_blocks(static_cast<const double*>(p) + off0, a.v.ts, step, nb, lane, s);
      };
      const int lb = lane / a.parts, lc = lane - lb * a.parts;
      const bool wanted = lane < qc && lb / a.per == c && lc >= y_first(lb) && lc < y_last(lb);
#pragma unroll 1
      for (int u = 0; u < t; ++u) {
        fetch(u);
        wait_flags(a.flags + kTile + u * 128, wanted, t - 1 - u);
        if (tid < PER * kNB) ys[tid] = tid < nb * kNB ? y_value(u, b0 * kNB + tid) : 0.0;
        __syncthreads();
        if (MIXED && f32) times_blocks<float, TRANS>(s, ys, lane, wave, acc);
        else times_blocks<double, TRANS>(s, ys, lane, wave, acc);
      }
      w = block_sum<TRANS>(acc, red, lane, wave);
      if constexpr (!ONE) {
        if (wave == 0) {
          store_through(a.part + (long)(2 * t + 1) * vec + c * ts + own * kNB + lane, w);
          stores_done();
          if (lane == 0) flag_put(a.flags + kTile + t * 128 + 64 + r, 1);
        }
        __syncthreads();
        continue;
      }
    }
    // B_t: the part's blocks in the triangle
    if (TRANS && own > b0) {
      const int skip = own - b0;
      off0 += skip * step;
      b0 += skip;
      nb -= skip;
    }
    if (!TRANS && own + 1 - b0 < nb) nb = own + 1 - b0;
    if (nb <= 0) continue;
    load_blocks(a.xinv + (long)m * ts * ts + off0, a.v.ts, step, nb, lane, s);
    const int i = b0 * kNB + tid;
    double x = tid < nb * kNB ? a.z[m * ts + i] : 0.0;
    if constexpr (ONE) {
      x -= w;
    } else if (t > 0) {
      wait_flags(a.flags + kTile + t * 128 + 64,
                 lane < qc && lane / a.parts >= b0 && lane / a.parts < b0 + nb, 0);
      if (tid < nb * kNB) x -= sum_parts(a.part + (long)(2 * t + 1) * vec + i, ts, 0, a.parts);
    }
    if (tid < PER * kNB) ys[tid] = x;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.0;
    times_blocks<double, TRANS>(s, ys, lane, wave, acc);
    const double y = block_sum<TRANS>(acc, red, lane, wave);
    if (wave == 0) {
      store_through(a.part + (long)2 * t * vec + c * ts + own * kNB + lane, y);
      if constexpr (ONE) a.z[m * ts + lane] = y;
      stores_done();
      if (lane == 0) flag_put(a.flags + kTile + t * 128 + r, 1);
    }
  }
  // The last work-group leaves the flags as it found them.
  if (tid == 0) sh = atomicAdd(a.flags + kExit, 1) == (int)gridDim.x - 1;
  __syncthreads();
  if (!sh) return;
  for (int e = tid; e < 128 * mt; e += 256) a.flags[kTile + e] = 0;
  if (tid == 0) a.flags[kClaim] = a.flags[kExit] = 0;
}

int strip_parts(int ts) { return (ts / kNB + 3) / 4; }

template <bool TRANS, bool MIXED, int PER>
void launch(const TrsvArgs& a, hipStream_t s) {
  static const int slots = [] {  // by the first thread that comes here; others wait for it
    int dev = 0, cus = 0, occ = 1;
    EXA_HIP(hipGetDevice(&dev));
    EXA_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    EXA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_trsv_flow<TRANS, MIXED, PER>, 256, 0));
    return cus * (occ > 0 ? occ : 1);
  }();
  const long tasks = PER == 1 ? a.v.mt : (long)a.q * a.parts * (2 * a.v.mt - 1) + a.v.mt;
  hipLaunchKernelGGL((k_trsv_flow<TRANS, MIXED, PER>), dim3((unsigned)(tasks < slots ? tasks : slots)), dim3(256), 0, s,
                     a);
  EXA_HIP(hipGetLastError());
}

template <bool TRANS>
void launch_trans(const TrsvArgs& a, hipStream_t s) {
  if (a.q == 1) {
    if (a.v.prec) launch<TRANS, true, 1>(a, s);
    else launch<TRANS, false, 1>(a, s);
  } else {
    if (a.v.prec) launch<TRANS, true, 4>(a, s);
    else launch<TRANS, false, 4>(a, s);
  }
}

}  // namespace

long trsv_part_doubles(int mt, int ts) { return 2L * mt * strip_parts(ts) * ts; }
long trsv_flags(int mt) { return kTile + 128L * mt; }

void launch_trsv(const TileView& v, const double* xinv, double* z, int trans, double* part, int* flags,
                 hipStream_t s) {
  TrsvArgs a;
  a.v = v;
  a.xinv = xinv;
  a.z = z;
  a.part = part;
  a.flags = flags;
  a.q = v.ts / kNB;
  a.parts = strip_parts(v.ts);
  a.per = (a.q + a.parts - 1) / a.parts;
  if (v.ts % kNB || a.q < 1 || a.q > 16 || v.mt < 1 || !xinv || !part || !flags)
    throw std::invalid_argument("trsv: tile size or scratch");
  if (trans) launch_trans<true>(a, s);
  else launch_trans<false>(a, s);
}

}  // namespace exa
