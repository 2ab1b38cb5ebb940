// C-ABI plumbing shared by every entry point: error recording and launch checks.
#include <stdarg.h>
#include <stdio.h>

#include <algorithm>
#include <atomic>
#include <string>

#include "gdn_common.h"

namespace {
thread_local std::string g_last_error;
}

namespace zgdn {

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

int check_launch(const char* what) {
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(ZGDN_EHIP, "%s: kernel launch failed: %s", what, hipGetErrorString(err));
  g_last_error.clear();
  return ZGDN_OK;
}

int device_cus() {
  constexpr int MAX_DEVICES = 64;
  static std::atomic<int> cus[MAX_DEVICES];
  int dev = 0, n = 256;
  if (hipGetDevice(&dev) != hipSuccess) return n;
  const bool kept = dev >= 0 && dev < MAX_DEVICES;
  if (kept) {
    const int v = cus[dev].load(std::memory_order_relaxed);
    if (v > 0) return v;
  }
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 256;
  n = std::max(1, n);
  if (kept) cus[dev].store(n, std::memory_order_relaxed);
  return n;
}

}  // namespace zgdn

extern "C" const char* zgdn_last_error(void) { return g_last_error.c_str(); }

extern "C" int zgdn_abi_version(void) { return 2; }
