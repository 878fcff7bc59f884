// Thread-local error message + launch checking for the C ABI.
#include <stdarg.h>
#include <stdio.h>

#include <mutex>

#include "common.h"

namespace {
thread_local char g_err[512] = "";
}

namespace wz {

int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(WZ_ELAUNCH, "%s: launch failed: %s", what, hipGetErrorString(e));
  return WZ_OK;
}

}  // namespace wz

extern "C" const char* wz_last_error(void) { return g_err; }

namespace wz {
// Compute units of the current device (cached per device; 256 on MI355X).
int cu_count() {
  static int cached[kMaxDevices] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// Lets `kernel` be launched with `bytes` of dynamic LDS on the current device.  Past 64 KB the
// runtime wants hipFuncAttributeMaxDynamicSharedMemorySize, which belongs to the current device's
// function: it is raised once per device and size, one thread at a time so that a smaller
// request never overwrites a larger one.
int allow_lds_of(const char* what, const void* kernel, size_t bytes, LdsGrant& grant) {
  if (bytes <= 64 * 1024) return WZ_OK;
  int dev = -1;
  const bool known = hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices;
  if (known && int(bytes) <= grant.bytes[dev].load(std::memory_order_acquire)) return WZ_OK;
  static std::mutex mu;
  std::lock_guard<std::mutex> lock(mu);
  if (known && int(bytes) <= grant.bytes[dev].load(std::memory_order_relaxed)) return WZ_OK;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)) != hipSuccess)
    return set_error(WZ_ELAUNCH, "%s: %zu bytes of LDS refused", what, bytes);
  if (known) grant.bytes[dev].store(int(bytes), std::memory_order_release);
  return WZ_OK;
}
}  // namespace wz

extern "C" int wz_device_info(int* cu_count, int* xcd_count) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return wz::set_error(WZ_EINVAL, "wz_device_info: no device");
  hipDeviceProp_t p;
  if (hipGetDeviceProperties(&p, dev) != hipSuccess)
    return wz::set_error(WZ_EINVAL, "wz_device_info: hipGetDeviceProperties failed");
  if (cu_count) *cu_count = p.multiProcessorCount;
  if (xcd_count) *xcd_count = 8;
  return WZ_OK;
}
