// The few runtime calls that pcx_xfer.hip makes, over host memory: copies are done
// when they are issued, events are always complete.
#pragma once
#include <cstddef>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
typedef int* hipStream_t;
typedef int* hipEvent_t;
constexpr unsigned hipHostMallocPortable = 1, hipEventDisableTiming = 2;

extern int g_fail_copies;                       // copies that fail from now on
extern int g_pinned;                            // pinned allocations alive

inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++g_pinned;
  return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void* p) {
  --g_pinned;
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = static_cast<int*>(std::malloc(4)); return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (g_fail_copies) return hipErrorUnknown;
  std::memcpy(d, s, n);
  return hipSuccess;
}
