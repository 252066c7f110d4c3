// The dynamic LDS limit of a kernel (beyond 64 KB a launch needs it raised).  The limit belongs to a device: a call site
// raises it before its launches on a device until that has been done once.  Threads launch side by side (the composites
// give the interpreter lock back), so a device is noted only behind the call that raises the limit: a second thread that
// comes meanwhile raises it again, which changes nothing, instead of launching without it.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace mega {

// `seen`: the call site's own mask of devices; kernels: every kernel that the site launches
template <typename... Kernels>
static inline void raise_lds_limit(uint64_t* seen, int bytes, Kernels... kernels) {
  int d = 0;
  if (hipGetDevice(&d) != hipSuccess) {
    (void)hipGetLastError();
    d = 0;
  }
  const uint64_t bit = 1ull << (d & 63);
  if (__atomic_load_n(seen, __ATOMIC_ACQUIRE) & bit) return;
  const void* const all[] = {(const void*)kernels...};
  for (const void* k : all) (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  __atomic_fetch_or(seen, bit, __ATOMIC_RELEASE);
}

}  // namespace mega
