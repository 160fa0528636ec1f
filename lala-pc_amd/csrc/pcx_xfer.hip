// pcx_xfer.hip -- large results from the device into pageable host memory.
//
// A caller's result arrays are fresh memory as a rule: the copy into them is
// bound by their page faults and by one core's copy speed (24 MB took 3.0 ms,
// while the link moves 57 GB/s), not by the link.  Here the caller and a few
// workers that live for the call each carry a share of the bytes through two
// pinned slots of their own, one filled by the device while the other is copied
// out.  (The other direction, from arrays a program has already written, is
// faster through the runtime: 24 MB in 0.9 ms, and 1.0 this way.)
//
// The slots (kThreads * 2 * kSlot bytes) are one pool for the process, freed with the
// last engine.  Their allocation takes 0.9 ms, which a copy of a few megabytes does not
// win back: they are made once copies of kWorth bytes have gone the runtime's way, so
// that a program that makes an engine, reads its results and drops it pays for none.
// A copy that finds the pool in use by another thread takes the runtime's path.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

#include "pcx_xfer.h"

namespace {

// Reading 24 MB into fresh arrays took 1.26, 1.25 and 1.21 ms with 3, 6 and 8
// threads (3.0 through the runtime): the page faults share one lock.  Slots of
// 512 and 256 KB took 1.4 and 2.0.
constexpr int kThreads = 4;
constexpr size_t kSlot = (size_t)1 << 20;
constexpr size_t kWorth = (size_t)32 << 20;     // what they save, about 26 us a megabyte, by then
constexpr size_t kShare = (size_t)1 << 20;      // bytes a further thread is worth starting for

struct Pool {
  std::mutex use;                               // held for the length of one copy
  std::mutex life;                              // users, and the slots' life
  int users = 0;
  uint8_t* slots = nullptr;
  size_t waited = 0;                            // bytes of large copies before there were slots
  hipEvent_t ev[2 * kThreads] = {};
  int device = -1;                              // the events' device
};
Pool g_pool;

void drop_events() {
  for (hipEvent_t& e : g_pool.ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  g_pool.device = -1;
}

// Slots and events for `device` (the current one), if copies like this one of `bytes`
// are worth them; the caller holds `use`.
bool ready(int device, size_t bytes) {
  if (!g_pool.slots && (g_pool.waited += std::min(bytes, kWorth)) <= kWorth) return false;
  if (!g_pool.slots &&
      hipHostMalloc(reinterpret_cast<void**>(&g_pool.slots), 2 * kThreads * kSlot, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    g_pool.slots = nullptr;
    return false;
  }
  if (g_pool.device != device) {
    drop_events();
    for (hipEvent_t& e : g_pool.ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        e = nullptr;
        drop_events();
        return false;
      }
    g_pool.device = device;
  }
  return true;
}

// Bytes [at, at + n) of the result, which lies in two arrays one after the other.
struct Dest {
  uint8_t* a;
  size_t na;                                    // bytes of the first
  uint8_t* b;
  void put(size_t at, const uint8_t* src, size_t n) const {
    const size_t first = at < na ? std::min(n, na - at) : 0;
    if (first) std::memcpy(a + at, src, first);
    if (n > first) std::memcpy(b + (at + first - na), src + first, n - first);
  }
};

// Thread t's share [at, end) through its two slots.
hipError_t carry_out(int t, const Dest& dst, const uint8_t* src, size_t at, size_t end, hipStream_t st) {
  auto issue = [&](size_t from, int i) {
    hipError_t he = hipMemcpyAsync(g_pool.slots + (2 * t + i) * kSlot, src + from, std::min(kSlot, end - from),
                                   hipMemcpyDeviceToHost, st);
    if (he == hipSuccess) he = hipEventRecord(g_pool.ev[2 * t + i], st);
    return he;
  };
  if (at >= end) return hipSuccess;
  hipError_t he = issue(at, 0);
  for (int i = 0; he == hipSuccess && at < end; at += kSlot, i ^= 1) {
    if (at + kSlot < end) he = issue(at + kSlot, i ^ 1);
    const hipError_t we = hipEventSynchronize(g_pool.ev[2 * t + i]);
    if (he == hipSuccess) he = we;
    if (he == hipSuccess) dst.put(at, g_pool.slots + (2 * t + i) * kSlot, std::min(kSlot, end - at));
  }
  return he;
}

template <class F>
hipError_t share_out(size_t bytes, int device, F carry) {
  const int threads = (int)std::min<size_t>(kThreads, std::max<size_t>(1, bytes / kShare));
  const size_t share = (bytes / threads + 4095) & ~(size_t)4095;
  hipError_t got[kThreads];
  auto work = [&](int t) {
    if (t > 0) (void)hipSetDevice(device);
    got[t] = carry(t, std::min(bytes, t * share), t + 1 == threads ? bytes : std::min(bytes, (t + 1) * share));
  };
  std::thread th[kThreads];
  for (int t = 1; t < threads; ++t) {
    try {
      th[t] = std::thread(work, t);
    } catch (const std::exception&) {           // no thread or no memory for one: the caller carries this share too
      work(t);
    }
  }
  work(0);
  hipError_t he = got[0];
  for (int t = 1; t < threads; ++t) {
    if (th[t].joinable()) th[t].join();
    if (he == hipSuccess) he = got[t];
  }
  return he;
}

}  // namespace

namespace pcx_internal {

void xfer_acquire() {
  std::lock_guard<std::mutex> l(g_pool.life);
  ++g_pool.users;
}

void xfer_release() {
  std::lock_guard<std::mutex> l(g_pool.life);
  if (--g_pool.users > 0) return;
  std::lock_guard<std::mutex> u(g_pool.use);
  drop_events();
  if (g_pool.slots) (void)hipHostFree(g_pool.slots);
  g_pool.slots = nullptr;
  g_pool.waited = 0;
}

hipError_t copy_to_host(void* dst, size_t bytes, void* dst2, size_t bytes2, const void* src, int device,
                        hipStream_t st) {
  if (bytes + bytes2 >= kXferMin) {
    std::unique_lock<std::mutex> l(g_pool.use, std::try_to_lock);
    if (l.owns_lock() && ready(device, bytes + bytes2)) {
      const Dest to{static_cast<uint8_t*>(dst), bytes, static_cast<uint8_t*>(dst2)};
      const hipError_t he = share_out(bytes + bytes2, device, [&](int t, size_t at, size_t end) {
        return carry_out(t, to, static_cast<const uint8_t*>(src), at, end, st);
      });
      if (he != hipSuccess) (void)hipStreamSynchronize(st);   // nothing queued still writes the slots
      return he;
    }
  }
  hipError_t he = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
  if (he == hipSuccess && bytes2)
    he = hipMemcpyAsync(dst2, static_cast<const uint8_t*>(src) + bytes, bytes2, hipMemcpyDeviceToHost, st);
  return he == hipSuccess ? hipStreamSynchronize(st) : he;
}

}  // namespace pcx_internal
