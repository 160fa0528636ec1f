// pcx_formula.hip -- PC's is_extractable over formula trees.
//
// A formula's postorder nodes (include/pcx_model.h) are interpreted with a stack
// of int2: intervals for terms, {ask, nask} for formulas (PC's Formula::ask /
// nask, include/lala/formula.hpp; the arithmetic of the terms' projections over
// int32 bounds whose extremes are the infinities).  A formula not asked clears
// its store's flag, and a store whose flag is clear is not asked further (PC's
// loop returns at the first formula not asked).
//
// Two kernels share the interpreter:
//  - k_formula_lanes: a wave takes one formula for 64 stores, over their
//    interleaved copy (variable v of a group's 64 stores is one run of 512
//    bytes).  Nodes are scalar loads, the node kind a scalar branch, a variable
//    one coalesced load, and the stack lies in LDS.  What bounds it: the copy's
//    bytes from L2 and the latency of a node.
//  - k_formula_ask: a thread per (store, formula), for few stores (their lanes
//    would be idle) and few formulas (the copy would take longer).  Every variable is a gather and every lane follows its own
//    nodes, the stack in scratch memory.
// 50,000 formulas on 512 stores of 12,500 variables, half of them solutions:
// 0.78 ms a thread per pair, 0.18 ms in lanes (and 0.02 for the copy).  On 16, 64
// and 2,000 solutions the whole call took 0.62, 0.69 and 5.3 ms a thread per pair,
// 0.61, 0.63 and 1.4 in lanes (0.4 of it the host's check of the trees, then).
#include "../../include/pcx_model.h"
#include "pcx_device.h"

#include <algorithm>

namespace pcx {

namespace tree {
constexpr int32_t kMinf = INT32_MIN, kInf = INT32_MAX;
__device__ __forceinline__ bool inf(i64 v) { return v == kMinf || v == kInf; }
__device__ __forceinline__ int32_t sat(i64 v) { return v <= kMinf ? kMinf : v >= kInf ? kInf : (int32_t)v; }
// a bound of a sum: the infinity it leans to wins over the other
__device__ __forceinline__ int32_t add(i64 a, i64 b, i64 first) {
  if (a == first || b == first) return (int32_t)first;
  if (inf(a)) return (int32_t)a;
  if (inf(b)) return (int32_t)b;
  return sat(a + b);
}
__device__ __forceinline__ int32_t neg(i64 a) { return a == kMinf ? kInf : a == kInf ? kMinf : (int32_t)-a; }
__device__ __forceinline__ int sgn(i64 a) { return (a > 0) - (a < 0); }
__device__ __forceinline__ i64 mul(i64 a, i64 b) {
  if (a == 0 || b == 0) return 0;
  if (inf(a) || inf(b)) return sgn(a) * sgn(b) > 0 ? kInf : kMinf;
  return a * b;
}
__device__ __forceinline__ i64 div(int kind, i64 a, i64 b) {
  if (inf(a)) return sgn(a) * sgn(b) > 0 ? kInf : kMinf;
  if (inf(b)) return 0;
  i64 q = a / b;                                   // truncated
  const i64 r = a - q * b;
  if (kind == PCX_FT_FDIV) { if (r != 0 && ((r < 0) != (b < 0))) --q; }
  else if (kind == PCX_FT_CDIV) { if (r != 0 && ((r < 0) == (b < 0))) ++q; }
  else if (kind == PCX_FT_EDIV) { if (r < 0) q += b > 0 ? -1 : 1; }
  return q;
}
}  // namespace tree

// A stack whose top is in registers; the rest is wherever `Rest` keeps it.
template <class Rest>
struct TreeStack {
  Rest rest;
  int sp = 0;
  int2 top = make_int2(0, 0);
  __device__ __forceinline__ void push(int2 v) {
    if (sp > 0) rest.put(sp - 1, top);
    top = v;
    ++sp;
  }
  __device__ __forceinline__ int2 under() const { return rest.get(sp - 2); }   // below the top
  __device__ __forceinline__ void fold(int2 v) { top = v; --sp; }              // the two upper ones become v
};

// Formula nodes [j, end) on a store read through `var`; the value it leaves.
template <class Stack, class Var>
__device__ __forceinline__ int2 interpret(const int4* __restrict__ nodes, int64_t j, int64_t end, Stack& s, Var var) {
  using tree::add;
  using tree::div;
  using tree::mul;
  using tree::neg;
  using tree::sat;
  constexpr int32_t kTMinf = tree::kMinf, kTInf = tree::kInf;
  for (; j < end; ++j) {
    const int4 nd = nodes[j];
    switch (nd.x) {
      case PCX_FT_VAR: s.push(var(nd.y)); break;
      case PCX_FT_CONST: s.push(make_int2(nd.y, nd.y)); break;
      case PCX_FT_TRUE: s.push(make_int2(1, 0)); break;
      case PCX_FT_FALSE: s.push(make_int2(0, 1)); break;
      case PCX_FT_NEG: s.top = make_int2(neg(s.top.y), neg(s.top.x)); break;
      case PCX_FT_ABS: {
        const int2 a = s.top;
        if (a.x >= 0) break;
        s.top = a.y <= 0 ? make_int2(neg(a.y), neg(a.x)) : make_int2(0, max((int32_t)neg(a.x), a.y));
        break;
      }
      case PCX_FT_ADD: case PCX_FT_SUB: {
        const int2 a = s.under();
        int2 b = s.top;
        if (nd.x == PCX_FT_SUB) b = make_int2(neg(b.y), neg(b.x));
        s.fold(make_int2(add(a.x, b.x, kTMinf), add(a.y, b.y, kTInf)));
        break;
      }
      case PCX_FT_MUL: {
        const int2 a = s.under(), b = s.top;
        const i64 c0 = mul(a.x, b.x), c1 = mul(a.x, b.y), c2 = mul(a.y, b.x), c3 = mul(a.y, b.y);
        s.fold(make_int2(sat(min(min(c0, c1), min(c2, c3))), sat(max(max(c0, c1), max(c2, c3)))));
        break;
      }
      case PCX_FT_TDIV: case PCX_FT_FDIV: case PCX_FT_CDIV: case PCX_FT_EDIV: {
        const int2 a = s.under(), b = s.top;
        int2 r = make_int2(kTMinf, kTInf);
        if (!(b.x <= 0 && 0 <= b.y)) {
          const i64 c0 = div(nd.x, a.x, b.x), c1 = div(nd.x, a.x, b.y), c2 = div(nd.x, a.y, b.x),
                    c3 = div(nd.x, a.y, b.y);
          r = make_int2(sat(min(min(c0, c1), min(c2, c3))), sat(max(max(c0, c1), max(c2, c3))));
        }
        s.fold(r);
        break;
      }
      case PCX_FT_MIN: case PCX_FT_MAX: {
        const int2 a = s.under(), b = s.top;
        s.fold(nd.x == PCX_FT_MIN ? make_int2(min(a.x, b.x), min(a.y, b.y))
                                  : make_int2(max(a.x, b.x), max(a.y, b.y)));
        break;
      }
      case PCX_FT_LE: case PCX_FT_LT: case PCX_FT_EQ: case PCX_FT_NE: {
        const int2 l = s.under(), r = s.top;
        int2 t;
        if (nd.x == PCX_FT_LE) t = make_int2(l.y <= r.x, l.x > r.y);
        else if (nd.x == PCX_FT_LT) t = make_int2(l.y < r.x, l.x >= r.y);
        else {
          const int same = l.x == l.y && r.x == r.y && l.x == r.x;
          const int apart = l.y < r.x || r.y < l.x;
          t = nd.x == PCX_FT_EQ ? make_int2(same, apart) : make_int2(apart, same);
        }
        s.fold(t);
        break;
      }
      case PCX_FT_AND: case PCX_FT_OR: {
        const int n = nd.y;
        int all_a = 1, any_a = 0, all_n = 1, any_n = 0;
        for (int q = s.sp - n; q < s.sp; ++q) {
          const int2 v = q == s.sp - 1 ? s.top : s.rest.get(q);
          all_a &= v.x; any_a |= v.x; all_n &= v.y; any_n |= v.y;
        }
        const int2 r = nd.x == PCX_FT_AND ? make_int2(all_a, any_n) : make_int2(any_a, all_n);
        if (n == 0) {
          s.push(r);
        } else {                                   // the n upper ones become r
          s.top = r;
          s.sp -= n - 1;
        }
        break;
      }
      case PCX_FT_NOT: s.top = make_int2(s.top.y, s.top.x); break;
      case PCX_FT_EQUIV: case PCX_FT_XOR: {
        const int2 fm = s.under(), g = s.top;
        const int same = (fm.x & g.x) | (fm.y & g.y), differ = (fm.x & g.y) | (fm.y & g.x);
        s.fold(nd.x == PCX_FT_EQUIV ? make_int2(same, differ) : make_int2(differ, same));
        break;
      }
      case PCX_FT_LIT: {
        const int2 a = s.top;
        s.top = make_int2(!(a.x <= 0 && 0 <= a.y), a.x >= 0 && a.y <= 0);
        break;
      }
      case PCX_FT_PROP: {
        const int4 zn = nodes[j + 1];
        s.push(make_int2(entailed(nd.y, var(nd.z), var(nd.w), var(zn.y)) ? 1 : 0, 0));
        ++j;                                       // the PROP_Z node
        break;
      }
      default: break;                              // (k_trees_check let none through)
    }
  }
  return s.top;
}

namespace {

constexpr int kGroup = kWave;          // stores per group of the interleaved copy
constexpr int kPerWave = 8;            // formulas a wave asks per turn

struct PrivateRest {
  int2 s[kTreeDepth];
  __device__ __forceinline__ void put(int i, int2 v) { s[i] = v; }
  __device__ __forceinline__ int2 get(int i) const { return s[i]; }
};
struct LdsRest {
  int2* s;                             // [depth][64], this lane's column
  __device__ __forceinline__ void put(int i, int2 v) { s[i * kWave] = v; }
  __device__ __forceinline__ int2 get(int i) const { return s[i * kWave]; }
};

}  // namespace

// A thread per formula: verdict[0] = 1 where a formula is not well formed (known
// kinds, variables inside the store, ternary opcodes, a stack within the depth
// limit that ends with one value, offsets in order), verdict[1] = the deepest
// stack.  The host's check of 264,000 nodes took 0.4 ms of a 0.8 ms call.
__global__ __launch_bounds__(kBlock) void k_trees_check(const int4* __restrict__ nodes, int64_t n_nodes,
                                                        const int64_t* __restrict__ off, int64_t n_formulas,
                                                        int32_t nvars, int32_t* verdict) {
  const int64_t f = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  bool bad = false;
  int depth = 0, deepest = 0;
  if (f < n_formulas) {
    const int64_t beg = off[f], end = off[f + 1];
    bad = beg < 0 || end < beg || end > n_nodes;
    auto var_ok = [&](int32_t v) { return v >= 0 && v < nvars; };
    for (int64_t j = beg; !bad && j < end; ++j) {
      const int4 nd = nodes[j];
      int pop = 0;
      switch (nd.x) {
        case PCX_FT_VAR: bad = !var_ok(nd.y); break;
        case PCX_FT_CONST: case PCX_FT_TRUE: case PCX_FT_FALSE: break;
        case PCX_FT_NEG: case PCX_FT_ABS: case PCX_FT_NOT: case PCX_FT_LIT: pop = 1; break;
        case PCX_FT_ADD: case PCX_FT_SUB: case PCX_FT_MUL: case PCX_FT_TDIV: case PCX_FT_FDIV:
        case PCX_FT_CDIV: case PCX_FT_EDIV: case PCX_FT_MIN: case PCX_FT_MAX: case PCX_FT_LE: case PCX_FT_LT:
        case PCX_FT_EQ: case PCX_FT_NE: case PCX_FT_EQUIV: case PCX_FT_XOR: pop = 2; break;
        case PCX_FT_AND: case PCX_FT_OR:
          pop = nd.y;
          bad = pop < 0;
          break;
        case PCX_FT_PROP: {
          bad = j + 1 >= end || nd.y < 0 || nd.y >= kNumOps || !var_ok(nd.z) || !var_ok(nd.w);
          if (!bad) {
            const int4 zn = nodes[j + 1];
            bad = zn.x != PCX_FT_PROP_Z || !var_ok(zn.y);
          }
          ++j;
          break;
        }
        default: bad = true; break;
      }
      bad |= depth < pop;
      depth += 1 - pop;
      deepest = max(deepest, depth);
      bad |= depth > kTreeDepth;
    }
    bad |= depth != 1;
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) deepest = max(deepest, __shfl_xor(deepest, o, kWave));
  const bool any = __ballot(bad) != 0;
  if (lane_id() == 0) {
    if (any) atomicOr(&verdict[0], 1);
    atomicMax(&verdict[1], deepest);
  }
}

hipError_t launch_trees_check(const int4* nodes, int64_t n_nodes, const int64_t* off, int64_t n_formulas,
                              int64_t nvars, int32_t* verdict, hipStream_t stream) {
  if (n_formulas <= 0) return hipSuccess;
  k_trees_check<<<(unsigned)((n_formulas + kBlock - 1) / kBlock), kBlock, 0, stream>>>(nodes, n_nodes, off, n_formulas,
                                                                                      (int32_t)nvars, verdict);
  return hipGetLastError();
}

// Threads take chunks of kBlock formulas of one instance, chunk by chunk over
// all instances, so that a store not extractable is found early.
__global__ __launch_bounds__(kBlock) void k_formula_ask(const int4* __restrict__ nodes, const int64_t* __restrict__ off,
                                                        int64_t n_formulas, const int2* __restrict__ store,
                                                        int64_t nvars, int64_t n_inst, int32_t* ok) {
  const int64_t chunks = (n_formulas + kBlock - 1) / kBlock;
  const int64_t total = chunks * n_inst * kBlock;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += (int64_t)gridDim.x * kBlock) {
    const int64_t row = i / kBlock, k = row % n_inst;
    const int64_t f = (row / n_inst) * kBlock + (i - row * kBlock);
    if (f >= n_formulas || !__hip_atomic_load(&ok[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) continue;
    const int2* st = store + k * nvars;
    TreeStack<PrivateRest> s;
    const int2 r = interpret(nodes, off[f], off[f + 1], s, [&](int32_t v) { return st[v]; });
    if (!r.x) __hip_atomic_store(&ok[k], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Turns of kPerWave formulas for one group, turn by turn over all groups.
__global__ __launch_bounds__(kBlock) void k_formula_lanes(const int4* __restrict__ nodes,
                                                          const int64_t* __restrict__ off, int64_t n_formulas,
                                                          const int2* __restrict__ shadow, int64_t nvars,
                                                          int64_t n_inst, int32_t* ok, int depth) {
  extern __shared__ int2 s_stack[];                // [waves][depth][64]
  const int lane = lane_id(), wave = uni((int32_t)(threadIdx.x / kWave));
  const int64_t groups = (n_inst + kGroup - 1) / kGroup;
  const int64_t turns = (n_formulas + kPerWave - 1) / kPerWave * groups;
  TreeStack<LdsRest> s;
  s.rest.s = s_stack + (int64_t)wave * depth * kWave + lane;
  for (int64_t i = (int64_t)blockIdx.x * (kBlock / kWave) + wave; i < turns; i += (int64_t)gridDim.x * (kBlock / kWave)) {
    const int64_t g = i % groups, f0 = i / groups * kPerWave, k = g * kGroup + lane;
    bool live = k < n_inst && __hip_atomic_load(&ok[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    const bool was = live;
    const int2* st = shadow + g * nvars * kGroup + lane;
    for (int64_t f = f0; f < min(f0 + kPerWave, n_formulas) && __ballot(live); ++f) {
      s.sp = 0;
      // every lane interprets (the copy is padded to whole groups), so that the
      // stack stays uniform
      const int2 r = interpret(nodes, uni(off[f]), uni(off[f + 1]), s,
                               [&](int32_t v) { return st[(int64_t)v * kGroup]; });
      live = live && r.x != 0;
    }
    if (was && !live) __hip_atomic_store(&ok[k], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

hipError_t launch_formula_ask(const int4* nodes, const int64_t* off, int64_t n_formulas, const int2* store,
                              int64_t nvars, int64_t n_inst, int32_t* ok, hipStream_t stream) {
  if (n_inst <= 0 || n_formulas <= 0) return hipSuccess;
  int64_t grid = ((n_formulas + kBlock - 1) / kBlock) * n_inst;     // one workgroup per (chunk, instance)
  if (grid > 8192) grid = 8192;
  k_formula_ask<<<(unsigned)grid, kBlock, 0, stream>>>(nodes, off, n_formulas, store, nvars, n_inst, ok);
  return hipGetLastError();
}

hipError_t launch_formula_lanes(const int4* nodes, const int64_t* off, int64_t n_formulas, int depth,
                                const int2* shadow, int64_t nvars, int64_t n_inst, int32_t* ok, int cus,
                                hipStream_t stream) {
  if (n_inst <= 0 || n_formulas <= 0) return hipSuccess;
  if (depth < 1 || depth > kTreeDepth) return hipErrorInvalidValue;
  const int64_t groups = (n_inst + kGroup - 1) / kGroup;
  const int64_t turns = (n_formulas + kPerWave - 1) / kPerWave * groups;
  const int64_t blocks = (turns + kBlock / kWave - 1) / (kBlock / kWave);
  const unsigned grid = (unsigned)std::min<int64_t>(blocks, (int64_t)cus * 8);
  k_formula_lanes<<<grid, kBlock, (size_t)(kBlock / kWave) * depth * kWave * sizeof(int2), stream>>>(
      nodes, off, n_formulas, shadow, nvars, n_inst, ok, depth);
  return hipGetLastError();
}

}  // namespace pcx
