// pcx_device.h -- device helpers shared by the kernel sources: lanes and waves,
// store loads and meets.
#pragma once
#include "pcx_kernels.h"
#include "pcx_prop.h"

namespace pcx {

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

// Values the whole wave agrees on (work-item indices, descriptors read
// through them) moved to scalar registers: the compiler cannot prove a load
// from a uniform address returns a uniform value, and would otherwise keep
// them, and everything derived from them, in VGPRs.
__device__ __forceinline__ int32_t uni(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uni(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
template <class T>
__device__ __forceinline__ T* uni(T* p) { return reinterpret_cast<T*>(uni((int64_t)(uintptr_t)p)); }

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

// ---- store access policies ------------------------------------------------
// Agent scope (sweep kernels: ordered by kernel boundaries) or workgroup
// scope (persistent kernel: one workgroup owns an instance).
template <int SCOPE>
__device__ __forceinline__ u64 load_word(const void* p) {
  if constexpr (SCOPE == __HIP_MEMORY_SCOPE_AGENT) return *reinterpret_cast<const u64*>(p);
  else return __hip_atomic_load(reinterpret_cast<const u64*>(p), __ATOMIC_RELAXED, SCOPE);
}
__device__ __forceinline__ int2 as_itv(u64 v) {
  return make_int2((int32_t)(uint32_t)v, (int32_t)(uint32_t)(v >> 32));
}
__device__ __forceinline__ u64 itv_bits(int2 v) { return (u64)(uint32_t)v.x | ((u64)(uint32_t)v.y << 32); }

// Meet interval `n` into variable v, whose value was read as `cur`.
// Returns true when this call tightened a bound of v.
template <int SCOPE>
__device__ __forceinline__ bool meet_itv(int2* __restrict__ st, int32_t v, int2 cur, int2 n,
                                         bool& chg, bool& fail, int& nt) {
  bool t = false;
  if (n.x > cur.x) {
    const int old = __hip_atomic_fetch_max(&st[v].x, n.x, __ATOMIC_RELAXED, SCOPE);
    if (old < n.x) { t = true; ++nt; }
    if (n.x > cur.y) fail = true;          // cur.y >= current ub
  }
  if (n.y < cur.y) {
    const int old = __hip_atomic_fetch_min(&st[v].y, n.y, __ATOMIC_RELAXED, SCOPE);
    if (old > n.y) { t = true; ++nt; }
    if (n.y < cur.x) fail = true;
  }
  chg |= t;
  return t;
}

// AND mask `n` into word v, whose value was read as `cur`.
template <int SCOPE>
__device__ __forceinline__ bool meet_word(u64* __restrict__ st, int32_t v, u64 cur, u64 n,
                                          bool& chg, bool& fail, int& nt) {
  bool t = false;
  if ((cur & n) != cur) {
    const u64 old = __hip_atomic_fetch_and(&st[v], n, __ATOMIC_RELAXED, SCOPE);
    if ((old & n) != old) { t = true; ++nt; }
    if ((old & n) == 0) fail = true;       // the word is now empty
  }
  chg |= t;
  return t;
}

// The meets of one propagator with all of its atomics issued before the first
// result is looked at (one latency instead of up to six in a row, where the
// owner of the store waits for nothing else): which operands were tightened.
template <int SCOPE>
__device__ __forceinline__ void meet3_itv(int2* __restrict__ st, int32_t x, int32_t y, int32_t z, int2 X, int2 Y,
                                          int2 Z, int2 nx, int2 ny, int2 nz, bool& tx, bool& ty, bool& tz,
                                          bool& fail, int& nt) {
  int32_t ox = nx.x, px = nx.y, oy = ny.x, py = ny.y, oz = nz.x, pz = nz.y;   // "old" values that change nothing
  if (nx.x > X.x) ox = __hip_atomic_fetch_max(&st[x].x, nx.x, __ATOMIC_RELAXED, SCOPE);
  if (nx.y < X.y) px = __hip_atomic_fetch_min(&st[x].y, nx.y, __ATOMIC_RELAXED, SCOPE);
  if (ny.x > Y.x) oy = __hip_atomic_fetch_max(&st[y].x, ny.x, __ATOMIC_RELAXED, SCOPE);
  if (ny.y < Y.y) py = __hip_atomic_fetch_min(&st[y].y, ny.y, __ATOMIC_RELAXED, SCOPE);
  if (nz.x > Z.x) oz = __hip_atomic_fetch_max(&st[z].x, nz.x, __ATOMIC_RELAXED, SCOPE);
  if (nz.y < Z.y) pz = __hip_atomic_fetch_min(&st[z].y, nz.y, __ATOMIC_RELAXED, SCOPE);
  // a bound that passes the other one, as it was read (X.y >= the current ub)
  fail |= nx.x > nx.y || ny.x > ny.y || nz.x > nz.y || nx.x > X.y || nx.y < X.x || ny.x > Y.y || ny.y < Y.x ||
          nz.x > Z.y || nz.y < Z.x;
  const bool a = ox < nx.x, b = px > nx.y, c = oy < ny.x, d = py > ny.y, e = oz < nz.x, f = pz > nz.y;
  tx = a | b;
  ty = c | d;
  tz = e | f;
  nt += (int)a + (int)b + (int)c + (int)d + (int)e + (int)f;
}

}  // namespace pcx
