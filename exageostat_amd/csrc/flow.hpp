// Hand-over of finished data between the work-groups of one launch: data are
// written through to the device's coherence point (agent-scope stores), then
// a flag is released at agent scope; a waiting work-group polls the flag and
// acquires at agent scope before it reads.
#pragma once

#include "common.hpp"

namespace exa {

__device__ __forceinline__ int flag_get(const int* f) {
  return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Every wave's stores have left the wave; to be called before the barrier
// that precedes flag_set.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__host__ __device__ __forceinline__ void flag_set(int* f, int v) {
  __hip_atomic_store(f, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}
// The same for a counter whose writers have not seen each other's values: it
// never goes back, in whatever order their stores arrive.
__host__ __device__ __forceinline__ void flag_raise(int* f, int v) {
  __hip_atomic_fetch_max(f, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void store_through(T* p, T v) {
  typedef __attribute__((address_space(1))) T gT;
  __hip_atomic_store((gT*)(uintptr_t)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Hand-over without cache maintenance, where everything that is handed over
// is written with store_through and read with load_through: both act at the
// coherence point, so completed stores (stores_done) need no write-back of
// the L2 and the reader no invalidation of it (a fence of work-group scope
// keeps the compiler's order; the reader's loads are issued after a branch on
// the flag's value).  This rests on how gfx950 performs agent-scope accesses:
// the language's memory model asks for release and acquire at agent scope,
// which cost an L2 write-back and an invalidation per hand-over.
__device__ __forceinline__ void flag_put(int* f, int v) {
  __hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T load_through(const T* p) {
  typedef __attribute__((address_space(1))) const T gT;
  return __hip_atomic_load((gT*)(uintptr_t)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace exa
