// Memory that the wave kernels' FP64 atomics reach (host code).
#pragma once
#include <hip/hip_runtime_api.h>

namespace frg {

// k_su adds to dGamma with FP64 atomics of the memory side.  Those are sure to
// take effect in ordinary allocations of the device that runs the kernel; host
// and managed memory, fine-grained or uncached allocations (they carry flags) and
// buffers of another device are written with plain stores, by the general kernel.
inline bool takes_fp64_atomics(const hipPointerAttribute_t &a, int device) {
  return a.type == hipMemoryTypeDevice && !a.isManaged && a.device == device &&
         a.allocationFlags == hipDeviceMallocDefault;
}

}  // namespace frg
