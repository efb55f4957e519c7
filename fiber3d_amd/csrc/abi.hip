// Error reporting and version query of the libf3d C ABI.
#include <stdarg.h>

#include "common.h"

#include <atomic>

namespace f3d {

static thread_local char g_last_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
}

int num_cus() {
  static std::atomic<int> cached{0};
  int n = cached.load(std::memory_order_relaxed);
  if (n > 0) return n;
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess)
    return 256;
  n = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
  cached.store(n, std::memory_order_relaxed);
  return n;
}
}  // namespace f3d

extern "C" const char* f3d_last_error(void) { return f3d::g_last_error; }

extern "C" int f3d_abi_version(void) { return 100; }
