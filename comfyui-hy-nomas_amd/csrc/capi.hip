// Library-wide C-ABI plumbing: version, per-thread error text, HIP status translation.
#include <stdarg.h>
#include <stdio.h>

#include <atomic>

#include "hn_common.h"

namespace hn {

static thread_local char g_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

int hip_status(hipError_t e, const char* what) {
  if (e == hipSuccess) return HN_OK;
  set_error("%s: %s", what, hipGetErrorString(e));
  return HN_ERR_HIP;
}

// Compute units of the current device.
// The per-device cache may be filled by several host threads at once; they store the same value.
int cu_count() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

}  // namespace hn

extern "C" int hn_version(void) { return 200; }

extern "C" const char* hn_last_error(void) { return hn::g_error; }
