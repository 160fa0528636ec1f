// pcx_ask.hip -- entailment over a batch: which propagators of which instances
// are still open.
//
// A propagator is asked once.  Workgroups take chunks of an instance's
// propagators (so a few instances still fill the device), keep the answers as
// bits, one 64-bit word per wave and step, and count them; a scan turns the
// counts into places; the bits are then written out as table positions.  What
// bounds it: the three operand gathers of an ask.  (One workgroup per instance,
// asking once to count and again to write, took 102 + 170 us for 128 instances
// of 50,000 propagators.)
#include "pcx_device.h"

#include <algorithm>

namespace pcx {

namespace {
constexpr int kAskWords = kAskChunk / kWave;           // words of a chunk
constexpr int kAskWaves = kBlock / kWave;
}  // namespace

__global__ __launch_bounds__(kBlock) void k_ask_bits(Table t, const int2* __restrict__ store, int64_t nvars,
                                                     Subsets sub, int64_t n_props, int64_t n_inst, int64_t chunks,
                                                     AskWork w) {
  __shared__ int s_cnt;
  const int lane = lane_id(), wave = uni((int32_t)(threadIdx.x / kWave));
  for (int64_t i = blockIdx.x; i < n_inst * chunks; i += gridDim.x) {
    const int64_t k = i / chunks, c = i - k * chunks;
    const int64_t m = sub.off ? sub.off[k + 1] - sub.off[k] : n_props;
    const int32_t* idx = sub.off ? sub.idx + sub.off[k] : nullptr;
    const int2* st = store + k * nvars;
    if (threadIdx.x == 0) s_cnt = 0;
    __syncthreads();
    int cnt = 0;
    for (int s = wave; s < kAskWords; s += kAskWaves) {
      const int64_t q = c * kAskChunk + s * kWave + lane;
      bool open = false;
      if (q < m) {
        const int64_t p = idx ? (int64_t)idx[q] : q;
        const uint32_t xo = t.xo[p];
        open = !entailed((int)(xo >> kOpShift), st[xo & kVarMask], st[t.y[p]], st[t.z[p]]);
      }
      const unsigned long long word = __ballot(open);
      if (lane == 0) w.bits[i * kAskWords + s] = word;
      cnt += __builtin_popcountll(word);
    }
    // this chunk's share of the variables: is one of them empty
    const int64_t share = (nvars + chunks - 1) / chunks;
    bool e = false;
    for (int64_t v = c * share + threadIdx.x; v < min(nvars, (c + 1) * share); v += kBlock) e |= st[v].x > st[v].y;
    if (__ballot(e) && lane == 0) w.empty[k] = 1;
    if (lane == 0 && cnt) atomicAdd(&s_cnt, cnt);
    __syncthreads();
    if (threadIdx.x == 0) w.count[i] = s_cnt;
    __syncthreads();                                   // s_cnt is rewritten next
  }
}

// The same with the store staged in LDS first, for stores that fit and instances of
// more than one chunk (a call on 1,000 stores of 250 variables and 1,000 propagators,
// or of 12,500 variables and subsets of 50: 44 and 64 us without it, 49 and 70 with):
// the gathers then cost LDS cycles instead of L2 requests.  A workgroup takes a part of an
// instance's chunks, four words of a wave in flight together.
constexpr int kAskWide = 1024, kAskUnroll = 4;
__global__ __launch_bounds__(kAskWide) void k_ask_bits_lds(Table t, const int2* __restrict__ store, int64_t nvars,
                                                           Subsets sub, int64_t n_props, int64_t n_inst, int64_t chunks,
                                                           int64_t parts, AskWork w) {
  extern __shared__ u64 s_store[];
  __shared__ int s_cnt[2];                             // by chunk parity
  constexpr int kWaves = kAskWide / kWave;
  const int2* st = reinterpret_cast<const int2*>(s_store);
  const int lane = lane_id(), wave = uni((int32_t)(threadIdx.x / kWave));
  for (int64_t i = blockIdx.x; i < n_inst * parts; i += gridDim.x) {
    const int64_t k = i / parts, part = i - k * parts;
    const int64_t m = sub.off ? sub.off[k + 1] - sub.off[k] : n_props;
    const int32_t* idx = sub.off ? sub.idx + sub.off[k] : nullptr;
    const u64* g = reinterpret_cast<const u64*>(store + k * nvars);
    if (threadIdx.x < 2) s_cnt[threadIdx.x] = 0;
    bool e = false;
    for (int64_t v = threadIdx.x; v < nvars; v += kAskWide) {
      const u64 b = g[v];
      s_store[v] = b;
      e |= as_itv(b).x > as_itv(b).y;
    }
    if (part == 0 && __ballot(e) && lane == 0) w.empty[k] = 1;
    __syncthreads();                                   // the store is in
    const int64_t c1 = (part + 1) * chunks / parts;
    for (int64_t c = part * chunks / parts; c < c1; ++c) {
      int cnt = 0;
      static_assert(kAskWords == kWaves * kAskUnroll, "one round of words per chunk");
      uint32_t xo[kAskUnroll];
      int32_t y[kAskUnroll], z[kAskUnroll];
      bool in[kAskUnroll];
#pragma unroll
      for (int u = 0; u < kAskUnroll; ++u) {
        const int64_t q = c * kAskChunk + (u * kWaves + wave) * kWave + lane;
        in[u] = q < m;
        xo[u] = 0;
        y[u] = z[u] = 0;
        if (in[u]) {
          const int64_t p = idx ? (int64_t)idx[q] : q;
          xo[u] = t.xo[p];
          y[u] = t.y[p];
          z[u] = t.z[p];
        }
      }
#pragma unroll
      for (int u = 0; u < kAskUnroll; ++u) {
        const bool open = in[u] && !entailed((int)(xo[u] >> kOpShift), st[xo[u] & kVarMask], st[y[u]], st[z[u]]);
        const unsigned long long word = __ballot(open);
        if (lane == 0) w.bits[(k * chunks + c) * kAskWords + u * kWaves + wave] = word;
        cnt += __builtin_popcountll(word);
      }
      if (lane == 0 && cnt) atomicAdd(&s_cnt[c & 1], cnt);
      __syncthreads();
      if (threadIdx.x == 0) {
        w.count[k * chunks + c] = s_cnt[c & 1];
        s_cnt[c & 1] = 0;                              // (the next chunk adds to the other)
      }
    }
    __syncthreads();                                   // the store is replaced next
  }
}

// One workgroup: off[k] = open propagators of the instances before k (off[n_inst]
// the total), place[i] = those of the chunks before chunk i, over all instances.
constexpr int kScanThreads = 1024;
__global__ __launch_bounds__(kScanThreads) void k_ask_places(AskWork w, int64_t n_inst, int64_t chunks) {
  __shared__ int64_t s_part[kScanThreads / kWave];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t n = n_inst * chunks;
  int64_t base = 0;
  for (int64_t i0 = 0; i0 < n; i0 += kScanThreads) {   // the same trip count in every thread
    const int64_t i = i0 + threadIdx.x;
    const int64_t c = i < n ? w.count[i] : 0;
    int64_t incl = c;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int64_t v = __shfl_up((long long)incl, o, kWave);
      if (lane >= o) incl += v;
    }
    if (lane == kWave - 1) s_part[wave] = incl;
    __syncthreads();
    int64_t before = 0, total = 0;
#pragma unroll
    for (int j = 0; j < kScanThreads / kWave; ++j) {
      if (j < wave) before += s_part[j];
      total += s_part[j];
    }
    if (i < n) {
      const int64_t at = base + before + incl - c;
      w.place[i] = at;
      if (i % chunks == 0) w.off[i / chunks] = at;
    }
    base += total;
    __syncthreads();                                   // s_part is rewritten next
  }
  if (threadIdx.x == 0) w.off[n_inst] = base;
}

// The open propagators' table positions, ascending per instance, as far as `cap`.
__global__ __launch_bounds__(kBlock) void k_ask_write(Subsets sub, int64_t n_inst, int64_t chunks, AskWork w,
                                                      int32_t* __restrict__ out, int64_t cap) {
  __shared__ int s_at[kAskWords];
  static_assert(kAskWords == kWave, "one word per lane");
  const int lane = lane_id(), wave = uni((int32_t)(threadIdx.x / kWave));
  for (int64_t i = blockIdx.x; i < n_inst * chunks; i += gridDim.x) {
    const int64_t k = i / chunks, c = i - k * chunks;
    const int32_t* idx = sub.off ? sub.idx + sub.off[k] : nullptr;
    if (wave == 0) {                                   // where each word's entries start
      const int n = __builtin_popcountll(w.bits[i * kAskWords + lane]);
      int incl = n;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const int v = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += v;
      }
      s_at[lane] = incl - n;
    }
    __syncthreads();
    const int64_t place = w.place[i];
    for (int s = wave; s < kAskWords; s += kAskWaves) {
      const unsigned long long word = w.bits[i * kAskWords + s];
      if (!((word >> lane) & 1ull)) continue;
      const int64_t at = place + s_at[s] +
                         (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(word >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)word, 0));
      const int64_t q = c * kAskChunk + s * kWave + lane;
      if (at < cap) out[at] = idx ? idx[q] : (int32_t)q;
    }
    __syncthreads();                                   // s_at is rewritten next
  }
}

int64_t ask_chunks(int64_t most_props) { return std::max<int64_t>(1, (most_props + kAskChunk - 1) / kAskChunk); }

hipError_t launch_ask_bits(const Table& t, const int2* store, int64_t nvars, const Subsets& sub, int64_t n_props,
                           int64_t n_inst, int64_t chunks, const AskWork& w, int device, int cus,
                           hipStream_t stream) {
  if (n_inst <= 0) return hipSuccess;
  const size_t sm = (size_t)nvars * sizeof(u64);
  if (chunks > 1 && (int64_t)sm <= lds_store_cap(device)) {
    if (sm > 65536) {                   // more dynamic LDS than the default is asked for first
      const hipError_t fe = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_ask_bits_lds),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
      if (fe != hipSuccess) return fe;
    }
    // enough parts for two workgroups per compute unit, at most one per chunk
    const int64_t parts = std::min<int64_t>(chunks, std::max<int64_t>(1, (2 * (int64_t)cus + n_inst - 1) / n_inst));
    const unsigned grid = (unsigned)std::min<int64_t>(n_inst * parts, 1 << 20);
    k_ask_bits_lds<<<grid, kAskWide, sm, stream>>>(t, store, nvars, sub, n_props, n_inst, chunks, parts, w);
  } else {
    const unsigned grid = (unsigned)std::min<int64_t>(n_inst * chunks, 1 << 20);
    k_ask_bits<<<grid, kBlock, 0, stream>>>(t, store, nvars, sub, n_props, n_inst, chunks, w);
  }
  return hipGetLastError();
}

hipError_t launch_ask_places(int64_t n_inst, int64_t chunks, const AskWork& w, hipStream_t stream) {
  if (n_inst <= 0) return hipSuccess;
  k_ask_places<<<1, kScanThreads, 0, stream>>>(w, n_inst, chunks);
  return hipGetLastError();
}

hipError_t launch_ask_write(const Subsets& sub, int64_t n_inst, int64_t chunks, const AskWork& w, int32_t* out,
                            int64_t cap, hipStream_t stream) {
  if (n_inst <= 0 || cap <= 0) return hipSuccess;
  const unsigned grid = (unsigned)std::min<int64_t>(n_inst * chunks, 1 << 20);
  k_ask_write<<<grid, kBlock, 0, stream>>>(sub, n_inst, chunks, w, out, cap);
  return hipGetLastError();
}

}  // namespace pcx
