// pcx_chase.hip -- a full sweep of one store whose waves chase what they tighten.
//
// A plain sweep advances a chain of propagators by about one link: the launch,
// not the link, sets the pace.  Here a wave evaluates 64 propagators of the
// table, then -- in the same launch, without barriers -- the propagators adjacent
// to what they tightened, and so on until nothing it tightened is left, before
// it takes its next 64.  A lane holds one propagator's record (position and
// operands) in registers; the adjacency holds whole records, so the lane that
// loads a neighbour already has what the next step evaluates, and the neighbours
// beyond the idle lanes wait in the wave's ring.
//
// Soundness needs nothing of the order: every value read is an
// over-approximation of the store (bounds only shrink), the meets are atomics.
// The operands of a chase are read with device-scope loads, since other
// workgroups tighten them during the launch.  Neighbours that find the ring full are dropped: a sweep that
// tightened anything is followed by another one over the whole table, and only a
// sweep that tightened nothing -- which read one constant store -- ends the run.
// For the same reason a wave may stop: after kChaseLinks links of a launch it drops
// what it was chasing and only evaluates the rest of its propagators once, so that
// a launch ends (after about 10 ms of links) however slowly the store converges,
// and a store that another wave has failed is left within kChaseLook links.  The
// walk of an adjacency ends when the ring is full, and a variable named by many
// propagators (hub_degree: an objective, a makespan) is not walked at all.  (These
// limits cost 3%: the chases of 200,000 propagators 0.54 ms, 0.52 without them.)
//
// What bounds it: three dependent trips to memory a link (operands; meets;
// adjacency records; about 2.3 us together), and the longest chain of links.  It
// pays once most propagators are settled: a few plain sweeps come first (one
// fixpoint of 200,000 / 4,000,000 propagators with 1, 2, 4, 8 and 16 of them:
// 0.84 / 3.45, 0.83 / 3.20, 0.77 / 3.06, 0.76 / 3.46 and 0.79 / 4.19 ms; plain and
// marked sweeps alone 1.92 / 6.27).  Stores that settle in a few more sweeps need no
// chase, which takes longer the more it finds to do: eight sweeps up to a million
// propagators (chains of 6, 10, 20 and 200 in 1,000,000 with 4 / 8 / plain sweeps
// alone: 750 / 513 / 617, 850 / 600 / 647, 920 / 925 / 735 and 1,260 / 1,330 / 2,890
// us; in 500,000: 493 / 333 / 375, 540 / 452 / 391, 575 / 545 / 517 and 920 / 930 /
// 2,080), four beyond, where a plain sweep costs more (1,400,000, the same chains
// but the first: 1,098 / 800 / 1,411, then 1,210 / 1,280 / 2,202 with chains of 30,
// 1,533 / 1,700 / 5,092).  Between 350,000 and a million propagators, stores of 10 to
// 30 sweeps still take longer than by plain sweeps, by a third at most: a wave ends
// one chase before it takes its next 64, and each wave has several.  Early chases cut after 1 to 8 links instead
// of the plain sweeps took 1.1-1.4 / 4.4-7.7 ms; 2, 3 or 7 workgroups per compute
// unit and 16 lanes per variable measured the same, 4 lanes 0.87 / 3.2.
#include "pcx_device.h"

#include <algorithm>

namespace pcx {

namespace {

constexpr int kChaseWaves = kBlock / kWave;
constexpr int kChaseRing = 1024;       // records' positions waiting, per wave (a power of two)
constexpr int kChaseLanes = 8;          // lanes that walk one variable's adjacency
constexpr int kChaseVars = kWave / kChaseLanes;
constexpr int kChaseLinks = 4096;       // links a wave chases in one launch
constexpr int kChaseLook = 64;          // links between two looks at the store's failure

// The adjacency a wave walks at most: eight lanes take about 0.05 us an entry, and
// what is not walked costs a sweep of the table (5 us, and 0.03 for 1,000
// propagators).
int32_t hub_degree(int64_t n_props) { return (int32_t)(128 + n_props / 4096); }

}  // namespace

template <int D>
__global__ __launch_bounds__(kBlock) void k_sweep_chase(Table t, int2* st, int32_t s, InstFlags* f,
                                                        unsigned long long* tight,
                                                        const int32_t* __restrict__ adj_off,
                                                        const int4* __restrict__ adj, int32_t hub) {
  constexpr int AG = __HIP_MEMORY_SCOPE_AGENT;
  // Sweep s runs only if sweep s-1 tightened something and nothing failed.
  if (f->changed[(s - 1) & 1] != s - 1 || f->failed_at != kNoFail) return;
  __shared__ int32_t s_ring[kChaseWaves][kChaseRing];
  __shared__ int2 s_walk[kChaseWaves][3 * kWave];    // adjacency ranges of the step's tightened variables
  const int lane = lane_id(), wave = uni((int32_t)(threadIdx.x / kWave));
  int32_t* const ring = s_ring[wave];
  int2* const walk = s_walk[wave];
  auto below = [](unsigned long long m) {            // set lanes below this one
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
  };
  const int64_t n_waves = (int64_t)gridDim.x * kChaseWaves;
  bool chg = false, fail = false;
  int nt = 0, ne = 0, links = 0, pause = kChaseLook;
  for (int64_t base = ((int64_t)blockIdx.x * kChaseWaves + wave) * kWave; base < t.n; base += n_waves * kWave) {
    uint32_t head = 0, tail = 0;                     // the ring's entries, the same in every lane
    bool on = base + lane < t.n;
    uint32_t xo = 0;
    int32_t y = 0, z = 0;
    if (on) {
      const int64_t q = base + lane;
      xo = t.xo[q];
      y = t.y[q];
      z = t.z[q];
    }
    for (bool first = true; __ballot(on); first = false) {
      const int32_t x = (int32_t)(xo & kVarMask);
      bool tx = false, ty = false, tz = false;
      int2 ax = make_int2(0, 0), ay = ax, az = ax;
      if (on) {
        // The adjacency ranges come with the operands (one trip): most chases
        // are chains, where a link's next trip would wait for them.
        const u64* const w = reinterpret_cast<const u64*>(st);
        u64 wx, wy, wz;
        if (first) {                                 // as a plain sweep reads them
          wx = w[x];
          wy = w[y];
          wz = w[z];
        } else {
          wx = __hip_atomic_load(w + x, __ATOMIC_RELAXED, AG);
          wy = __hip_atomic_load(w + y, __ATOMIC_RELAXED, AG);
          wz = __hip_atomic_load(w + z, __ATOMIC_RELAXED, AG);
        }
        if (!first) {
          ax = make_int2(adj_off[x], adj_off[x + 1]);
          ay = make_int2(adj_off[y], adj_off[y + 1]);
          az = make_int2(adj_off[z], adj_off[z + 1]);
        }
        const int op = (int)(xo >> kOpShift);
        const int2 X = as_itv(wx), Y = as_itv(wy), Z = as_itv(wz);
        if (X.x > X.y || Y.x > Y.y || Z.x > Z.y) {
          fail = true;
        } else {
          int2 nx, ny, nz;
          deduce<D == kItvDiv>(op, X, Y, Z, nx, ny, nz);
          meet3_itv<AG>(st, x, y, z, X, Y, Z, nx, ny, nz, tx, ty, tz, fail, nt);
        }
        ne += !first;
        if (first) {
          if (tx) ax = make_int2(adj_off[x], adj_off[x + 1]);
          if (ty) ay = make_int2(adj_off[y], adj_off[y + 1]);
          if (tz) az = make_int2(adj_off[z], adj_off[z + 1]);
        }
      }
      const unsigned long long mx = __ballot(tx), my = __ballot(ty), mz = __ballot(tz);
      chg |= (mx | my | mz) != 0;
      if (__ballot(fail)) break;
      if (!first && ++links >= pause) {
        if (links >= kChaseLinks || __hip_atomic_load(&f->failed_at, __ATOMIC_RELAXED, AG) != kNoFail) break;
        pause = links + kChaseLook;
      }
      const int cx = __builtin_popcountll(mx), cy = cx + __builtin_popcountll(my);
      const int nv = cy + __builtin_popcountll(mz);
      if (tx) walk[below(mx)] = ax;
      if (ty) walk[cx + below(my)] = ay;
      if (tz) walk[cy + below(mz)] = az;
      on = false;
      for (int i0 = 0; i0 < nv; i0 += kChaseVars) {
        const int i = i0 + lane / kChaseLanes;
        int2 range = i < nv ? walk[i] : make_int2(0, 0);
        if (range.y - range.x > hub) range.y = range.x;
        for (int32_t a = range.x + (lane & (kChaseLanes - 1)); __ballot(a < range.y); a += kChaseLanes) {
          const bool got = a < range.y;
          int4 rec = make_int4(0, 0, 0, 0);
          if (got) rec = adj[a];
          const unsigned long long more = __ballot(got && on);
          if (got && on) {
            const uint32_t at = tail + (uint32_t)below(more);
            if (at - head < kChaseRing) ring[at & (kChaseRing - 1)] = rec.x;
          } else if (got) {
            on = true;
            xo = (uint32_t)rec.y;
            y = rec.z;
            z = rec.w;
          }
          if (!more) continue;
          tail = min(tail + (uint32_t)__builtin_popcountll(more), head + (uint32_t)kChaseRing);
          if (uni((int32_t)(tail - head)) == kChaseRing) {   // full: the rest is dropped
            i0 = nv;
            break;
          }
        }
      }
      if (tail != head) {                            // idle lanes take the oldest entries
        const unsigned long long idle = __ballot(!on);
        const uint32_t r = (uint32_t)below(idle);
        if (!on && r < tail - head) {
          const int32_t q = ring[(head + r) & (kChaseRing - 1)];
          on = true;
          xo = t.xo[q];
          y = t.y[q];
          z = t.z[q];
        }
        head += min(tail - head, (uint32_t)__builtin_popcountll(idle));
      }
    }
    if (__ballot(fail)) break;
    if (__hip_atomic_load(&f->failed_at, __ATOMIC_RELAXED, AG) != kNoFail) break;
  }
  const int sum = wave_sum(nt), evals = wave_sum(ne);
  const bool bf = __ballot(fail) != 0;
  if (lane == 0) {
    if (chg) f->changed[s & 1] = s;
    if (bf) __hip_atomic_store(&f->failed_at, s, __ATOMIC_RELAXED, AG);
    if (sum) atomicAdd(&tight[(blockIdx.x * kChaseWaves + wave) & (kTightSlots - 1)], (unsigned long long)sum);
    if (evals) atomicAdd((unsigned long long*)&f->marked_evals, (unsigned long long)evals);
  }
}

hipError_t launch_sweep_chase(const Table& t, int2* store, int32_t sweep, InstFlags* flags,
                              unsigned long long* tight, const int32_t* adj_off, const int4* adj, int dom, int cus,
                              hipStream_t stream) {
  if (t.n <= 0) return hipSuccess;
  const unsigned grid = (unsigned)std::min<int64_t>((t.n + kBlock - 1) / kBlock, (int64_t)cus * 4);
  const int32_t hub = hub_degree(t.n);
  switch (dom) {
    case kItv: k_sweep_chase<kItv><<<grid, kBlock, 0, stream>>>(t, store, sweep, flags, tight, adj_off, adj, hub); break;
    case kItvDiv: k_sweep_chase<kItvDiv><<<grid, kBlock, 0, stream>>>(t, store, sweep, flags, tight, adj_off, adj, hub); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace pcx
