// Library-level C ABI: version and per-thread error reporting; host queries shared by
// the launchers.
#include <atomic>
#include <string>

#include "ia_common.hpp"

namespace ia {

namespace {
thread_local std::string g_last_error;
}

void set_error(const std::string& msg) { g_last_error = msg; }

int fail(int code, const std::string& msg) {
  set_error(msg);
  return code;
}

int check_launch(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(IA_ERR_LAUNCH, std::string(what) + ": " + hipGetErrorString(e));
  return IA_OK;
}

int device_cus() {
  constexpr int kMaxCachedDevices = 64;
  static std::atomic<int> cached[kMaxCachedDevices];  // (concurrent first calls store the same value)
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 256;
  if (dev < kMaxCachedDevices) n = cached[dev].load(std::memory_order_relaxed);
  if (n > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
  if (dev < kMaxCachedDevices) cached[dev].store(n, std::memory_order_relaxed);
  return n;
}

}  // namespace ia

extern "C" {

const char* ia_last_error(void) { return ia::g_last_error.c_str(); }

int ia_version(void) { return 1; }

}  // extern "C"
