// Which buffers sp_compute_step_noalloc hands to the kernels that add with atomics.
#include <cstdio>

#include "atomic_memory.h"

static hipPointerAttribute_t attributes(hipMemoryType type, int device, int managed, unsigned flags) {
  hipPointerAttribute_t a{};
  a.type = type;
  a.device = device;
  a.isManaged = managed;
  a.allocationFlags = flags;
  return a;
}

int main() {
  using frg::takes_fp64_atomics;
  const bool ok = takes_fp64_atomics(attributes(hipMemoryTypeDevice, 0, 0, 0), 0) &&
                  takes_fp64_atomics(attributes(hipMemoryTypeDevice, 3, 0, 0), 3) &&
                  !takes_fp64_atomics(attributes(hipMemoryTypeDevice, 1, 0, 0), 0) &&  // another GPU's
                  !takes_fp64_atomics(attributes(hipMemoryTypeDevice, 0, 0, hipDeviceMallocFinegrained), 0) &&
                  !takes_fp64_atomics(attributes(hipMemoryTypeDevice, 0, 0, hipDeviceMallocUncached), 0) &&
                  !takes_fp64_atomics(attributes(hipMemoryTypeHost, 0, 0, 0), 0) &&
                  !takes_fp64_atomics(attributes(hipMemoryTypeManaged, 0, 1, 0), 0) &&
                  !takes_fp64_atomics(attributes(hipMemoryTypeDevice, 0, 1, 0), 0) &&
                  !takes_fp64_atomics(attributes(hipMemoryTypeUnregistered, 0, 0, 0), 0);
  std::printf(ok ? "ok\n" : "wrong\n");
  return ok ? 0 : 1;
}
