// Library-wide state: thread-local error text, ABI version, device queries.
#include "common.h"

#include <atomic>

namespace mi355q {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

// (asked several times on the way to a launch of a few microseconds: a look-up without a lock; two threads that find nothing store the same)
int device_cu_count() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int cus = cached[dev].load(std::memory_order_relaxed);
  if (cus == 0) {
    hipDeviceProp_t p;
    cus = (hipGetDeviceProperties(&p, dev) == hipSuccess && p.multiProcessorCount > 0) ? p.multiProcessorCount : 256;
    cached[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

}  // namespace mi355q

extern "C" const char* mi355q_last_error(void) { return mi355q::g_err; }
// bumped whenever an entry point changes its arguments: the Python binding refuses a library of another version
// (a stale build would be called with shifted arguments)
extern "C" int mi355q_abi_version(void) { return 5; }
