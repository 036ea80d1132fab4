// Version, error reporting and split planning of the C ABI.
#include <atomic>
#include <cstdarg>

#include "wn_common.h"

namespace wn {

namespace {
thread_local std::string g_last_error;
}

void set_error(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
}

void clear_error() { g_last_error.clear(); }

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: %s", what, hipGetErrorString(e));
    return WN_E_LAUNCH;
  }
  return WN_OK;
}

int device_cus() {
  static std::atomic<int> known[64];
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 0;
  if (dev < 64 && (cus = known[dev].load(std::memory_order_relaxed)) > 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  if (dev < 64) known[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

}  // namespace wn

extern "C" int wn_abi_version(void) { return WN_ABI_VERSION; }

extern "C" const char* wn_last_error(void) { return wn::g_last_error.c_str(); }
