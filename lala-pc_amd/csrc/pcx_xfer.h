// pcx_xfer.h -- large results from the device into pageable host memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace pcx_internal {
constexpr size_t kXferMin = (size_t)1 << 20;     // smaller copies take the runtime's path
// Every engine holds the pool of pinned slots between these two.
void xfer_acquire();
void xfer_release();
// bytes + bytes2 at `src` into dst and then dst2 (bytes2 may be 0), after what is
// queued on the current device's stream `st`; complete on return.
hipError_t copy_to_host(void* dst, size_t bytes, void* dst2, size_t bytes2, const void* src, int device,
                        hipStream_t st);
}  // namespace pcx_internal
