// pcx_adj.hip -- the adjacency of a table: for every variable the propagators that
// name it (each once), built on the device from the table it holds.
//
// Count, scan, place: a propagator adds one to each of its variables' counts, the
// counts are scanned into offsets, and each propagator takes a place in its
// variables' ranges with an atomic (so the order within a range is any; nothing
// depends on it).  Neighbouring propagators often share a variable that most of the
// table names, so the lanes that agree with the first one take their places with
// one atomic.  What bounds it: the atomics, 3 n returning ones to scattered counters.
// The first fixpoint of a network waits for this: the host's two passes over the
// table in random order took 3 ms at 200,000 propagators, 6 at 1 M and 60 at 4 M.
#include "pcx_device.h"

#include <algorithm>

namespace pcx {

namespace {

constexpr int kScanPer = 16;                          // counts per thread
constexpr int kScanTile = kBlock * kScanPer;
constexpr int kTopThreads = 1024;

// A place in v's range for every lane that is on.
__device__ __forceinline__ int32_t take(int32_t* __restrict__ at, int32_t v, bool on) {
  const unsigned long long active = __ballot(on);
  if (!active) return 0;
  const int first = __builtin_ctzll(active);
  const int32_t fv = __builtin_amdgcn_readlane(v, first);
  const unsigned long long same = __ballot(on && v == fv);
  int32_t got = 0;
  if (lane_id() == first) got = atomicAdd(&at[fv], (int)__builtin_popcountll(same));
  got = __builtin_amdgcn_readlane(got, first);
  if (on && v != fv) return atomicAdd(&at[v], 1);
  return got + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0));
}

// The places that propagator p's variables give it, each distinct one once.
template <class F>
__device__ __forceinline__ void each_variable(const Table& t, int64_t p, int32_t* __restrict__ at, F put) {
  const bool on = p < t.n;
  int32_t x = 0, y = 0, z = 0;
  if (on) {
    x = (int32_t)(t.xo[p] & kVarMask);
    y = t.y[p];
    z = t.z[p];
  }
  const bool oy = on && y != x, oz = on && z != x && z != y;
  const int32_t ix = take(at, x, on), iy = take(at, y, oy), iz = take(at, z, oz);
  if (on) put(ix);
  if (oy) put(iy);
  if (oz) put(iz);
}

__device__ __forceinline__ int32_t wave_scan(int32_t v) {   // inclusive
  const int lane = lane_id();
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int32_t u = __shfl_up(v, o, kWave);
    if (lane >= o) v += u;
  }
  return v;
}

// Exclusive scan over a workgroup of N threads; *total the sum.
template <int N>
__device__ __forceinline__ int32_t block_scan(int32_t v, int32_t* s_part, int32_t* total) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int32_t incl = wave_scan(v);
  if (lane == kWave - 1) s_part[wave] = incl;
  __syncthreads();
  int32_t before = 0, all = 0;
#pragma unroll
  for (int j = 0; j < N / kWave; ++j) {
    if (j < wave) before += s_part[j];
    all += s_part[j];
  }
  __syncthreads();                                    // s_part may be rewritten
  *total = all;
  return before + incl - v;
}

}  // namespace

__global__ __launch_bounds__(kBlock) void k_adj_count(Table t, int32_t* __restrict__ at) {
  each_variable(t, (int64_t)blockIdx.x * kBlock + threadIdx.x, at, [](int32_t) {});
}

__global__ __launch_bounds__(kBlock) void k_adj_place(Table t, int32_t* __restrict__ at, int32_t* __restrict__ adj) {
  const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  each_variable(t, p, at, [&](int32_t i) { adj[i] = (int32_t)p; });
}

// Sums of tiles of counts.
__global__ __launch_bounds__(kBlock) void k_adj_sums(const int32_t* __restrict__ at, int64_t nvars,
                                                     int32_t* __restrict__ sums) {
  __shared__ int32_t s_part[kBlock / kWave];
  const int64_t v0 = (int64_t)blockIdx.x * kScanTile;
  int32_t sum = 0, total;
  for (int i = 0; i < kScanPer; ++i) {
    const int64_t v = v0 + i * kBlock + threadIdx.x;
    if (v < nvars) sum += at[v];
  }
  block_scan<kBlock>(sum, s_part, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// The tiles' sums, scanned in place by one workgroup; off[nvars] the whole sum.
__global__ __launch_bounds__(kTopThreads) void k_adj_top(int32_t* __restrict__ sums, int64_t n_tiles,
                                                         int32_t* __restrict__ off, int64_t nvars) {
  __shared__ int32_t s_part[kTopThreads / kWave];
  int32_t base = 0;
  for (int64_t i0 = 0; i0 < n_tiles; i0 += kTopThreads) {   // the same trip count in every thread
    const int64_t i = i0 + threadIdx.x;
    int32_t total;
    const int32_t e = block_scan<kTopThreads>(i < n_tiles ? sums[i] : 0, s_part, &total);
    if (i < n_tiles) sums[i] = base + e;
    base += total;
  }
  if (threadIdx.x == 0) off[nvars] = base;
}

// Offsets of a tile's variables, also as the places to take next.
__global__ __launch_bounds__(kBlock) void k_adj_offsets(int32_t* __restrict__ at, int64_t nvars,
                                                        const int32_t* __restrict__ sums, int32_t* __restrict__ off) {
  __shared__ int32_t s_part[kBlock / kWave];
  int32_t base = sums[blockIdx.x];
  const int64_t v0 = (int64_t)blockIdx.x * kScanTile;
  for (int i = 0; i < kScanPer; ++i) {
    const int64_t v = v0 + i * kBlock + threadIdx.x;
    int32_t total;
    const int32_t e = base + block_scan<kBlock>(v < nvars ? at[v] : 0, s_part, &total);
    if (v < nvars) {
      off[v] = e;
      at[v] = e;
    }
    base += total;
  }
}

int64_t adj_scratch(int64_t nvars) { return nvars + (nvars + kScanTile - 1) / kScanTile; }

hipError_t launch_adjacency(const Table& t, int64_t nvars, int32_t* off, int32_t* adj, int32_t* scratch,
                            hipStream_t stream) {
  if (t.n <= 0 || nvars <= 0) return hipErrorInvalidValue;
  const int64_t tiles = (nvars + kScanTile - 1) / kScanTile;
  int32_t* const at = scratch;
  int32_t* const sums = scratch + nvars;
  const unsigned grid = (unsigned)((t.n + kBlock - 1) / kBlock);
  const hipError_t he = hipMemsetAsync(at, 0, nvars * sizeof(int32_t), stream);
  if (he != hipSuccess) return he;
  k_adj_count<<<grid, kBlock, 0, stream>>>(t, at);
  k_adj_sums<<<(unsigned)tiles, kBlock, 0, stream>>>(at, nvars, sums);
  k_adj_top<<<1, kTopThreads, 0, stream>>>(sums, tiles, off, nvars);
  k_adj_offsets<<<(unsigned)tiles, kBlock, 0, stream>>>(at, nvars, sums, off);
  k_adj_place<<<grid, kBlock, 0, stream>>>(t, at, adj);
  return hipGetLastError();
}

}  // namespace pcx
