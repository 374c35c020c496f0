// rt_xfer.h -- host arrays of doubles to and from device arrays of double or
// float (the state of a level, emma_rt_set_level / emma_rt_get_level).
#pragma once

#include <hip/hip_runtime.h>

#include <stddef.h>

namespace emma {

// A device made current for a scope.  Streams, events and allocations belong to
// the device that is current when they are made, and a context's calls may come
// from a thread that has another one.
class DeviceScope {
 public:
  explicit DeviceScope(int device) {
    int now = device;
    if (hipGetDevice(&now) == hipSuccess && now != device && hipSetDevice(device) == hipSuccess) before_ = now;
  }
  ~DeviceScope() {
    if (before_ >= 0) (void)hipSetDevice(before_);
  }
  DeviceScope(const DeviceScope&) = delete;
  DeviceScope& operator=(const DeviceScope&) = delete;

 private:
  int before_ = -1;
};

// one array: n values, device storage float (f32) or double.  floor > 0 (to
// the device, f32): a value at or above it that rounds below it becomes
// floor_up, the smallest float at or above it.
struct XferPart {
  void* dev;
  void* host;
  size_t n;
  int f32;
  float floor_up;
  double floor;
};
constexpr int kMaxXferParts = 24;

// Both wait for the work queued on the stream before and return with the copy
// done.  Callable from several threads, whatever their current device; the
// staging memory is shared by all callers, bounded (32 MiB), and all but 16 MiB
// of it released with the last xfer_release().
hipError_t xfer_to_host(int device, hipStream_t s, const XferPart* parts, int np);
hipError_t xfer_to_device(int device, hipStream_t s, const XferPart* parts, int np);
// a user of the staging memory comes (a context is made) and goes
void xfer_retain();
void xfer_release();

}  // namespace emma
