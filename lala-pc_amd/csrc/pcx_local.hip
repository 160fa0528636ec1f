// pcx_local.hip -- fixpoints of stores that fit in a workgroup's LDS.
//
// One workgroup owns an instance from its first evaluation to its fixpoint in
// one launch, with the store and a bitmap of the propagators to evaluate in
// LDS.  The table and the adjacency are read from memory (every instance of a
// batch shares them, so they stay in L2).
//
// Rounds: (B) the workgroup evaluates what is marked -- walking the bitmap in
// table order while much of the table is marked (dense), else from the round's
// list -- clearing each mark before its operands are read, and lists each
// tightened variable once (a bitmap of variables).  (C) After a barrier, groups
// of lanes walk the adjacency of the listed variables and mark the instance's
// propagators, each new mark also listed for the next round.  A list that
// overflows makes the next round dense; variables that overflow theirs, or that are
// more than a sixteenth of the propagators, mark every propagator; an instance of a
// batch of intervals that has kManyRounds such rounds in a row is left to sweeps, too.
//
// Chase, once few marks are left: each wave propagates its share of them
// without barriers.  A lane holds one propagator's record (position, operands)
// in registers, the wave evaluates its 64, and walks the adjacency of what
// they tightened, four variables at a time.  The adjacency holds whole records,
// so a lane that finds a new mark already has what the next step evaluates; a
// second mark of the same lane goes to the wave's stack, from which idle lanes
// refill.  The bitmap keeps a propagator on one wave only.  A stack that
// overflows leaves the mark in the bitmap and sends the instance back to a
// dense round when the waves are done.
//
// Why this ends at the fixpoint: a propagator whose operand was tightened has
// its bit set afterwards (in a round by phase C, in a chase by the wave that
// tightened it), and whoever clears a bit reads the operands after that.  LDS
// operations of a wave complete in order, so a wave that finds a bit already
// set knows that its holder has not read the operands yet.  When no bit is set,
// every propagator was evaluated on operands that have not changed since.
//
// Hubs: a variable that many propagators name (hub_degree: an objective, a
// makespan) is not walked.  Its tightening marks everything, for a dense round; an
// instance that tightens hubs again and again (more than kHubRounds times) is left,
// kLocalLeft, to sweeps of its whole table, which then do less than its walks and
// lists.  (A chain of 200 links that each raise a variable of 3,200 propagators took
// 21 ms for 256 stores where lanes walked its adjacency, 0.99 in full sweeps.)
//
// A launch gives an instance kLocalLinks rounds and chase steps.  One that is not
// at its fixpoint then stays unsettled (settled_at < 0), its store as far as it
// came, and the host launches again: the instance goes on with every propagator
// marked, and its counts with it.  So a launch ends (4,096 steps of a chase take 6
// ms) however slowly a store converges.
//
// What bounds it: the depth of the propagation times the latency of one link
// (operands and meets in LDS, the adjacency from L2, and the instructions of one
// evaluation, which a lone wave issues one by one).
#include "pcx_device.h"

#include <algorithm>

namespace pcx {

namespace {

// Tightened variables listed per round, or per wave and chase step: at most
// three for each of a wave's 64 propagators.
constexpr int vars_of(int block) { return block / kWave * 192 > 1024 ? block / kWave * 192 : 1024; }
constexpr int kLocalList = 2048;       // propagators listed per round
constexpr int kWalkLanes = 16;         // lanes that walk one variable's adjacency in a chase
constexpr int kWalkVars = kWave / kWalkLanes;
constexpr int kChasePerWave = 8;         // marks a wave chases at most when a chase starts
constexpr int kLocalLinks = 4096;      // rounds and chase steps of an instance in one launch
constexpr int64_t kLocalStatic = 256;  // static LDS of the kernel (counters), at most
// Listed variables whose walks would take longer than another dense round, which
// is what shallow networks have most of: 4,096 stores with 2,000 propagators that
// settle in 6, 11 and 100 rounds took 224, 307 and 1,033 us without this line, 197,
// 273 and 1,014 with it (an eighth 198, 270, 1,019; a thirty-second 198, 287, 1,046;
// full sweeps 193, 276, 2,771); 1,000 with 16,000 propagators, 200 deep, 990, 974
// (986; 1,065; 5,931).
constexpr int kManyShift = 4, kManyLeast = 64;
// Such rounds in a row before an instance is left to sweeps, whose rounds are shorter
// and which more workgroups run at a time (256 / 1,000 stores in which chains of 100
// rise by one a round, 4,000 and 16,000 propagators: 0.77 / 2.36 and 2.40 / 14.8 ms
// here, 0.64 / 1.31 and 2.13 / 8.6 left after 4, 0.66 / 1.47 and 2.25 / 9.2 after 8,
// 0.71 / 1.67 and 2.39 / 10.1 after 16, 0.60 / 1.16 and 2.05 / 8.0 in sweeps alone;
// generated networks, 1 to 200 deep: the same).  Counted in LDS: in registers every
// wave's count cost a spill and 2 to 5% of the chases.
constexpr int kManyRounds = 4;
constexpr int kHubRounds = 2;          // dense rounds after hubs before the instance is left
// Propagators of a variable from which on it is a hub: a walk of 16 lanes takes about
// 0.025 us an entry, a sweep by the workgroup 1.3 us and 0.001 a propagator.
int32_t hub_degree(int64_t n_props) { return (int32_t)(96 + std::min<int64_t>(n_props / 32, 1024)); }
constexpr int32_t kResumeMax = 1 << 30;  // rounds a resumed run is taken to have had, at most (they are counted in 32 bits)

// Workgroups of 1,024 threads (batches that leave compute units idle: the
// dense rounds are then as wide as one unit allows) or 512 (larger batches:
// other instances fill the unit).
constexpr int kWide = 1024, kNarrow = 512;

int64_t bitmap_bytes(int64_t bits) { return (bits + 63) / 64 * 8; }

// store | marked propagators | listed variables | tightened variables |
// two lists (16-bit entries while the table's positions fit) | adjacency offsets
int64_t local_bytes(int64_t nvars, int64_t n_props, int block, bool offsets) {
  const int64_t entry = n_props <= 65536 ? 2 : 4;
  return nvars * 8 + bitmap_bytes(n_props) + bitmap_bytes(nvars) + vars_of(block) * 2 +
         2 * entry * kLocalList + (offsets ? (nvars + 1) * 4 : 0);
}


}  // namespace

bool local_fits(int device, int64_t nvars, int64_t n_props) {
  return n_props > 0 && n_props < ((int64_t)1 << 30) && nvars <= 65536 &&
         local_bytes(nvars, n_props, kWide, false) + kLocalStatic <= lds_store_cap(device);
}

// The adjacency with each propagator's table entry beside its position.
__global__ __launch_bounds__(kBlock) void k_adj_records(Table t, const int32_t* __restrict__ adj, int64_t n,
                                                        int4* __restrict__ rec) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int32_t q = adj[i];
  rec[i] = make_int4(q, (int32_t)t.xo[q], t.y[q], t.z[q]);
}

hipError_t launch_adj_records(const Table& t, const int32_t* adj, int64_t n, int4* rec, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  k_adj_records<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, stream>>>(t, adj, n, rec);
  return hipGetLastError();
}

namespace {
__device__ __forceinline__ long long wave_sum64(long long v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  return v;
}
}  // namespace

template <int D, int B>
constexpr int local_min_waves() { return B == kNarrow && D != kItvDiv ? 6 : 1; }

// OFFL: the adjacency offsets are copied to LDS.
template <int D, int B, class PT, bool OFFL>
__global__ __launch_bounds__(B, (local_min_waves<D, B>())) void k_local(Table t, LocalJob job) {
  constexpr int WG = __HIP_MEMORY_SCOPE_WORKGROUP;
  constexpr int kWaves = B / kWave;
  constexpr int kLocalVars = vars_of(B);
  constexpr int kStack = kLocalList / kWaves;        // marks on a wave's stack: its share of a list
  extern __shared__ u64 s_dyn[];
  __shared__ int32_t s_slot, s_fail, s_chg, s_steps;
  __shared__ int32_t s_empty;                        // empty as loaded: no round writes it, a late wave may still read it
  __shared__ int32_t s_ntv[2], s_n[2], s_over[2];    // by parity of the round
  __shared__ int32_t s_out;                          // a wave ran out of steps
  __shared__ int32_t s_many;                         // rounds in a row that marked everything (the first thread's)
  __shared__ int32_t s_hub, s_chub;                  // a hub was tightened in a round, in a chase (a
                                                     // late wave reads the one while the other is set);
                                                     // s_hub also ends an instance that is left
  __shared__ unsigned long long s_sum[3];
  const int tid = threadIdx.x, lane = lane_id(), wave = uni(tid / kWave);
  const int32_t V = (int32_t)job.nvars, P = (int32_t)t.n;
  const int32_t W = (P + 31) >> 5, VW = (V + 31) >> 5;
  u64* const st64 = s_dyn;
  int2* const st = reinterpret_cast<int2*>(s_dyn);
  uint32_t* const bm = reinterpret_cast<uint32_t*>(s_dyn + V);
  uint32_t* const vbm = bm + ((P + 63) >> 6) * 2;
  uint16_t* const tv = reinterpret_cast<uint16_t*>(vbm + ((V + 63) >> 6) * 2);
  PT* const lists = reinterpret_cast<PT*>(tv + kLocalVars);
  int32_t* const s_off = reinterpret_cast<int32_t*>(lists + 2 * kLocalList);
  const int32_t nadj = job.adj_vars;                 // variables with adjacency offsets
  if constexpr (OFFL)
    for (int32_t v = tid; v <= nadj; v += B) s_off[v] = job.adj_off[v];
  auto off = [&](int32_t v) {
    if constexpr (OFFL) return s_off[v];
    else return job.adj_off[v];
  };

  for (;;) {
    if (tid == 0) s_slot = job.queue ? atomicAdd(job.queue, 1) : 0;
    __syncthreads();
    const int32_t slot = s_slot;
    if (slot >= job.n_inst) return;                  // the same value in every wave
    const int32_t k = job.order ? job.order[slot] : slot;
    InstFlags* const f = job.flags + k;
    const bool soa = job.lb != nullptr;
    // (settled in an earlier launch of a run that goes on: nothing is left to do)
    bool start_failed = !soa && (f->failed_at != kNoFail || (job.resume && f->settled_at >= 0));
    const int32_t r0 = job.resume ? uni(min(max(f->done_at, 0), kResumeMax)) : 0;
    const uint32_t* const mrow = job.member ? job.member + (int64_t)k * job.words : nullptr;
    u64* const gst = soa ? nullptr : reinterpret_cast<u64*>(job.store) + (int64_t)k * V;
    auto member_word = [&](int32_t w) {              // every propagator of the instance
      if (mrow) return mrow[w];
      return (w == W - 1 && (P & 31)) ? (1u << (P & 31)) - 1u : ~0u;
    };
    if (tid == 0) { s_fail = 0; s_empty = 0; s_chg = 0; s_steps = 0; s_ntv[0] = s_ntv[1] = 0; s_n[0] = s_n[1] = 0; s_over[r0 & 1] = 1; s_over[(r0 & 1) ^ 1] = 0; s_out = s_hub = s_chub = s_many = 0; }
    if (tid < 3) s_sum[tid] = 0;
    __syncthreads();                                 // s_slot is read; the counters are set
    if (!start_failed) {
      bool empty = false;
      if (soa) {
        for (int32_t v = tid; v < V; v += B) {
          const int2 b = make_int2(job.lb[v], job.ub[v]);
          st[v] = b;
          empty |= b.x > b.y;
        }
      } else {
        for (int32_t v = tid; v < V; v += B) st64[v] = gst[v];
      }
      for (int32_t w = tid; w < W; w += B) bm[w] = member_word(w);
      for (int32_t w = tid; w < VW; w += B) vbm[w] = 0;
      if (empty) s_empty = 1;
      __syncthreads();
      start_failed = s_empty != 0;
    }

    int32_t failed_at = start_failed ? -1 : kNoFail, r = r0;
    const int32_t r_end = r0 + kLocalLinks;
    bool unsettled = false;
    int hubs = 0;                                    // rounds and chases that tightened one
    int nt0 = 0, nt = 0;                             // (a launch's share fits: kLocalLinks bounds it)
    int ne = 0;                                      // evaluations after round 0
    // Evaluate one propagator on the LDS store; which operands it tightened.
    bool fail = false;
    int tight = 0;
    bool tx = false, ty = false, tz = false;
    auto eval = [&](uint32_t xo, int32_t y, int32_t z) {
      const int32_t x = (int32_t)(xo & kVarMask);
      const int op = (int)(xo >> kOpShift);
      const u64 wx = load_word<WG>(st64 + x), wy = load_word<WG>(st64 + y), wz = load_word<WG>(st64 + z);
      tx = ty = tz = false;
      if constexpr (D == kBits) {
        if (!wx || !wy || !wz) { fail = true; return; }
        bool c = false;
        u64 nxw, nyw, nzw;
        deduce_bits(op, wx, wy, wz, nxw, nyw, nzw);
        tx = meet_word<WG>(st64, x, wx, nxw, c, fail, tight);
        ty = meet_word<WG>(st64, y, wy, nyw, c, fail, tight);
        tz = meet_word<WG>(st64, z, wz, nzw, c, fail, tight);
      } else {
        const int2 X = as_itv(wx), Y = as_itv(wy), Z = as_itv(wz);
        if (X.x > X.y || Y.x > Y.y || Z.x > Z.y) { fail = true; return; }
        int2 nxv, nyv, nzv;
        deduce<D == kItvDiv>(op, X, Y, Z, nxv, nyv, nzv);
        meet3_itv<WG>(st, x, y, z, X, Y, Z, nxv, nyv, nzv, tx, ty, tz, fail, tight);
      }
    };
    auto set_mark = [&](int32_t q) {                 // true when the bit was clear
      const uint32_t bit = 1u << (q & 31);
      if (mrow && !(mrow[q >> 5] & bit)) return false;
      return !(__hip_atomic_fetch_or(&bm[q >> 5], bit, __ATOMIC_RELAXED, WG) & bit);
    };
    // After a hub, between two barriers that every wave passes: everything is marked
    // and nothing listed, so that round r is a dense one.
    auto mark_everything = [&]() {
      for (int32_t w = tid; w < W; w += B) bm[w] = member_word(w);
      for (int32_t w = tid; w < VW; w += B) vbm[w] = 0;
      if (tid == 0) {
        s_n[0] = s_n[1] = 0;
        s_ntv[0] = s_ntv[1] = 0;
        s_over[r & 1] = 1;
        s_over[(r & 1) ^ 1] = 0;
        s_hub = s_chub = 0;
        s_steps = 0;
      }
    };
    while (!start_failed) {
      unsettled = r >= r_end;
      if (unsettled) break;
      // ---- round r: (B)
      const int cur = r & 1, nx = cur ^ 1;
      PT* const list = lists + cur * kLocalList;
      PT* const next = lists + nx * kLocalList;
      {
        auto note = [&](int32_t v) {
          const uint32_t bit = 1u << (v & 31);
          if (__hip_atomic_fetch_or(&vbm[v >> 5], bit, __ATOMIC_RELAXED, WG) & bit) return;
          const int at = __hip_atomic_fetch_add(&s_ntv[cur], 1, __ATOMIC_RELAXED, WG);
          if (at < kLocalVars) tv[at] = (uint16_t)v;
        };
        // Dense: a wave's 64 positions are two bitmap words, which only it
        // reads and clears in this phase.  The next entry is in flight while
        // one is evaluated.
        const bool dense = s_over[cur] != 0;
        const int32_t n = dense ? P : s_n[cur];
        bool on1 = false;
        uint32_t xo1 = 0;
        int32_t y1 = 0, z1 = 0;
        auto fetch = [&](int32_t i) {
          int32_t p = i;
          if (dense) {
            const uint32_t word = i < P ? bm[i >> 5] : 0u;
            if ((lane & 31) == 0 && word) bm[i >> 5] = 0;
            on1 = (word >> (i & 31)) & 1u;
          } else {
            on1 = i < n;
            if (on1) {
              p = (int32_t)list[i];
              __hip_atomic_fetch_and(&bm[p >> 5], ~(1u << (p & 31)), __ATOMIC_RELAXED, WG);
            }
          }
          if (on1) { xo1 = t.xo[p]; y1 = t.y[p]; z1 = t.z[p]; }
        };
        tight = 0;
        fetch(tid);
        for (int32_t i = tid; i - lane < n; i += B) {
          const bool on = on1;
          const uint32_t xo = xo1;
          const int32_t y = y1, z = z1;
          fetch(i + B);
          if (on) {
            eval(xo, y, z);
            ne += r > 0;
            if (tx) note((int32_t)(xo & kVarMask));
            if (ty) note(y);
            if (tz) note(z);
          }
        }
        if (r == 0) nt0 = tight; else nt += tight;
      }
      if (fail) s_fail = 1;
      __syncthreads();                               // the tightened variables are listed
      const int ntv = s_ntv[cur];
      if (ntv && tid == 0) s_chg = r + 1;
      if (s_fail) { failed_at = r; break; }
      if (!ntv) break;                               // quiet: the fixpoint
      // ---- (C)
      if (tid == 0) { s_ntv[nx] = 0; s_n[cur] = 0; s_over[cur] = 0; }
      if (ntv > min(kLocalVars, max(P >> kManyShift, kManyLeast))) {   // many, or some were lost: mark everything
        for (int32_t w = tid; w < W; w += B) bm[w] = member_word(w);
        for (int32_t w = tid; w < VW; w += B) vbm[w] = 0;
        if (tid == 0) {
          s_over[nx] = 1;
          if (job.sweeps && ++s_many > kManyRounds) s_hub = kHubRounds + 1;
        }
      } else {
        if (tid == 0) s_many = 0;
        // sixteen lanes per variable when that takes one pass, else eight
        const int lg = ntv * 16 <= B ? 4 : 3;
        const int sub = tid & ((1 << lg) - 1);
        for (int i = tid >> lg; i < ntv; i += B >> lg) {
          const int32_t v = (int32_t)tv[i];
          if (sub == 0) __hip_atomic_fetch_and(&vbm[v >> 5], ~(1u << (v & 31)), __ATOMIC_RELAXED, WG);
          const int32_t a0 = off(v), e = off(v + 1);
          if (e - a0 > job.hub) { s_hub = 1; continue; }
          for (int32_t a = a0 + sub; a < e; a += 1 << lg) {
            const int32_t q = job.adj[a].x;
            if (!set_mark(q)) continue;
            const int at = __hip_atomic_fetch_add(&s_n[nx], 1, __ATOMIC_RELAXED, WG);
            if (at < kLocalList) next[at] = (PT)q;
            else s_over[nx] = 1;
          }
        }
      }
      ++r;
      __syncthreads();                               // every mark is set and listed
      if (s_hub) {
        hubs += s_hub;
        unsettled = hubs > kHubRounds;
        if (unsettled) break;
        __syncthreads();                             // every wave has read it
        mark_everything();
        __syncthreads();
        continue;
      }
      const int marks = s_n[nx];
      if (s_over[nx] || marks > kChasePerWave * kWaves) continue;
      // ---- chase: each wave its share of the marks (the next round's list,
      // which no wave writes; the stacks take the other list's room)
      PT* const stack = list + wave * kStack;
      uint16_t* const wv = tv + wave * 192;          // what this wave's step tightened
      auto below = [](unsigned long long m) {        // set lanes below this one
        return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
      };
      int top = 0, steps = 0;                        // the same in every lane
      auto push = [&](bool on, int32_t p) {          // every lane of the wave calls it
        const unsigned long long m = __ballot(on);
        if (!m) return;
        const int at = top + below(m);
        if (on && at < kStack) stack[at] = (PT)p;
        top += __builtin_popcountll(m);
        if (top > kStack) {                          // the marks stay in the bitmap
          top = kStack;
          if (lane == 0) s_over[cur] = 1;
        }
      };
      tight = 0;
      int32_t q = -1, y = 0, z = 0;
      uint32_t xo = 0;
      {
        const int i = wave + kWaves * lane;
        if (i < marks) {
          q = (int32_t)next[i];
          xo = t.xo[q];
          y = t.y[q];
          z = t.z[q];
        }
      }
      for (; steps < r_end - r && __ballot(q >= 0); ++steps) {
        const int32_t stop = __hip_atomic_load(&s_fail, __ATOMIC_RELAXED, WG);   // arrives with the operands
        tx = ty = tz = false;
        if (q >= 0) {
          __hip_atomic_fetch_and(&bm[q >> 5], ~(1u << (q & 31)), __ATOMIC_RELAXED, WG);
          eval(xo, y, z);
          ++ne;
        }
        if (__ballot(fail || stop != 0)) {
          if (lane == 0) s_fail = 1;
          break;
        }
        // walk the adjacency of what was tightened, kWalkVars variables at a time
        const unsigned long long mx = __ballot(tx), my = __ballot(ty), mz = __ballot(tz);
        const int cx = __builtin_popcountll(mx), cy = cx + __builtin_popcountll(my);
        const int nv = cy + __builtin_popcountll(mz);
        if (tx) wv[below(mx)] = (uint16_t)(xo & kVarMask);
        if (ty) wv[cx + below(my)] = (uint16_t)y;
        if (tz) wv[cy + below(mz)] = (uint16_t)z;
        int32_t nq = -1, ny = 0, nz = 0;
        uint32_t nxo = 0;
        for (int i0 = 0; i0 < nv; i0 += kWalkVars) {
          const int i = i0 + lane / kWalkLanes;
          const int32_t v = i < nv ? (int32_t)wv[i] : -1;
          int32_t a = v >= 0 ? off(v) : 0;
          int32_t e = v >= 0 ? off(v + 1) : 0;
          if (e - a > job.hub) { s_chub = 1; e = a; }
          a += lane & (kWalkLanes - 1);
          while (__ballot(a < e)) {
            bool fresh = false;
            int4 rec = make_int4(-1, 0, 0, 0);
            if (a < e) {
              rec = job.adj[a];
              fresh = set_mark(rec.x);
            }
            push(fresh && nq >= 0, rec.x);
            if (fresh && nq < 0) { nq = rec.x; nxo = (uint32_t)rec.y; ny = rec.z; nz = rec.w; }
            a += kWalkLanes;
          }
        }
        q = nq;
        xo = nxo;
        y = ny;
        z = nz;
        if (top > 0) {                               // idle lanes take marks off the stack
          const unsigned long long idle = __ballot(q < 0);
          const int rank = below(idle);
          if (q < 0 && rank < top) {
            q = (int32_t)stack[top - 1 - rank];
            xo = t.xo[q];
            y = t.y[q];
            z = t.z[q];
          }
          top -= min(top, (int)__builtin_popcountll(idle));
        }
      }
      nt += tight;
      if (__ballot(q >= 0) && lane == 0) s_out = 1;  // (or it failed)
      if (lane == 0) __hip_atomic_fetch_max(&s_steps, steps, __ATOMIC_RELAXED, WG);
      const bool wave_changed = __ballot(tight != 0) != 0;
      __syncthreads();                               // every wave is done
      r += s_steps;                                  // steps count as rounds
      if (wave_changed && lane == 0) s_chg = r;
      if (s_fail) { failed_at = r; break; }
      const bool hub = s_chub != 0;
      hubs += hub;
      unsettled = s_out != 0 || hubs > kHubRounds;
      if (unsettled || !(hub || s_over[cur])) break; // no marks left anywhere: the fixpoint
      // Marks that found a stack full: a dense round (of the parity r has now).
      __syncthreads();                               // every wave has read the flags
      if (hub) {
        mark_everything();
        __syncthreads();
        continue;
      }
      if (tid == 0) {
        s_steps = 0;
        s_n[0] = s_n[1] = 0;
        s_ntv[0] = s_ntv[1] = 0;
        s_over[r & 1] = 1;
        s_over[(r & 1) ^ 1] = 0;
      }
      __syncthreads();
    }
    // ---- results
    const long long sums[3] = {wave_sum64(nt0), wave_sum64(nt), wave_sum64(ne)};
    if (lane == 0)
      for (int i = 0; i < 3; ++i)
        if (sums[i]) __hip_atomic_fetch_add(&s_sum[i], (unsigned long long)sums[i], __ATOMIC_RELAXED, WG);
    if (soa) {
      for (int32_t v = tid; v < V && !start_failed; v += B) {
        const int2 b = st[v];
        job.lb[v] = b.x;
        job.ub[v] = b.y;
      }
    } else if (!start_failed) {
      for (int32_t v = tid; v < V; v += B) gst[v] = st64[v];
    }
    __syncthreads();                                 // the sums and s_chg are in
    if (tid == 0) {
      const int32_t last = s_chg - 1;                // the last round that tightened something
      if (soa && !job.resume) *f = InstFlags{{-2, -1}, failed_at, r, 0, 0, -1, {-1, -1}};
      if (last >= 0) f->changed[last & 1] = last;
      if (!start_failed) {
        f->failed_at = failed_at;
        f->done_at = r;
        f->marked_evals += (int64_t)s_sum[2];
        f->settled_at = !unsettled ? r : hubs > kHubRounds ? kLocalLeft : -1;
      }
      if (job.tight) {
        const int at = slot & (kTightSlots - 1);
        if (s_sum[0]) atomicAdd(&job.tight[at], s_sum[0]);
        if (s_sum[1]) atomicAdd(&job.tight[kTightSlots + at], s_sum[1]);
      }
    }
    if (!job.queue) return;
    __syncthreads();                                 // s_slot and the sums are rewritten next
  }
}

namespace {

template <int D, int B, class PT, bool OFFL>
hipError_t launch_local_d(const Table& t, const LocalJob& job, int cus, hipStream_t stream) {
  const size_t sm = (size_t)local_bytes(job.nvars, t.n, B, OFFL);
  LocalJob j = job;
  j.hub = hub_degree(t.n);
  auto* const kernel = &k_local<D, B, PT, OFFL>;
  if (sm > 65536) {                     // more dynamic LDS than the default is asked for first
    const hipError_t fe = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
    if (fe != hipSuccess) return fe;
  }
  int per_cu = 1;
  if (job.n_inst > cus &&
      (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, B, sm) != hipSuccess || per_cu < 1))
    per_cu = 1;
  const unsigned grid = (unsigned)std::min<int64_t>(job.n_inst, (int64_t)cus * per_cu);
  kernel<<<grid, B, sm, stream>>>(t, j);
  return hipGetLastError();
}

template <int D, class PT>
hipError_t launch_local_p(const Table& t, const LocalJob& job, int device, int cus, hipStream_t stream) {
  if (job.n_inst > cus) return launch_local_d<D, kNarrow, PT, false>(t, job, cus, stream);
  if (local_bytes(job.nvars, t.n, kWide, true) + kLocalStatic <= lds_store_cap(device))
    return launch_local_d<D, kWide, PT, true>(t, job, cus, stream);
  return launch_local_d<D, kWide, PT, false>(t, job, cus, stream);
}

template <int D>
hipError_t launch_local_t(const Table& t, const LocalJob& job, int device, int cus, hipStream_t stream) {
  return t.n <= 65536 ? launch_local_p<D, uint16_t>(t, job, device, cus, stream)
                      : launch_local_p<D, int32_t>(t, job, device, cus, stream);
}

}  // namespace

hipError_t launch_local(const Table& t, const LocalJob& job, int dom, int device, int cus, hipStream_t stream) {
  if (job.n_inst <= 0) return hipSuccess;
  if ((job.lb == nullptr) == (job.store == nullptr) || !job.adj_off || job.adj_vars > job.nvars ||
      ((job.lb || !job.queue) && job.n_inst != 1))
    return hipErrorInvalidValue;
  switch (dom) {
    case kItv: return launch_local_t<kItv>(t, job, device, cus, stream);
    case kItvDiv: return launch_local_t<kItvDiv>(t, job, device, cus, stream);
    case kBits: return launch_local_t<kBits>(t, job, device, cus, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pcx
