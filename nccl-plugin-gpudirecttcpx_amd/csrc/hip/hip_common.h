// Shared by the translation units of the HIP layer: error plumbing and per-device helpers.
#ifndef TCPXU_HIP_COMMON_H_
#define TCPXU_HIP_COMMON_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "tcpx_unpack_hip.h"

namespace tcpxu {

constexpr int kMaxDevices = 64;

void set_error(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
int use_device(int device);            // hipSetDevice + cache properties
int device_compute_units(int device);  // valid after use_device
bool device_known(int device);         // use_device has been there

// The blocks that tcpxuMappedAlloc has given out, as one caller last saw them: it looks an address up in its own copy
// and takes a new one only when blocks have come or gone since.
struct MappedView {
  struct Block {
    uintptr_t dev, host;
    size_t bytes;
  };
  uint64_t generation = 0;
  std::vector<Block> blocks;  // by device address
};
// The host's address of `bytes` bytes at a device address inside one of those blocks, or null.
const void* mapped_host_address(MappedView* view, const void* dev, size_t bytes);

// Engine calls arrive on threads that belong to somebody else (NCCL's proxy thread calls tcpxTest, which may have
// to relaunch the kernel): the calling thread's current device is put back when the call returns.
class DeviceScope {
 public:
  explicit DeviceScope(int device) {
    if (hipGetDevice(&saved_) != hipSuccess) saved_ = -1;
    if (saved_ != device || !device_known(device)) rc_ = use_device(device);
    if (saved_ == device) saved_ = -1;  // nothing to put back
  }
  ~DeviceScope() {
    if (saved_ >= 0) (void)hipSetDevice(saved_);
  }
  int rc() const { return rc_; }
  DeviceScope(const DeviceScope&) = delete;
  DeviceScope& operator=(const DeviceScope&) = delete;

 private:
  int saved_ = -1;
  int rc_ = TCPXU_SUCCESS;
};

}  // namespace tcpxu

// A failing HIP call returns the "unhandled device error" code, as CUCHECK does in the reference
// (src/misc/cuda_checks.h:38-49); nothing in this layer calls exit().
#define TCPXU_HIP(call)                                                                              \
  do {                                                                                               \
    hipError_t e_ = (call);                                                                          \
    if (e_ != hipSuccess) {                                                                          \
      ::tcpxu::set_error("%s:%d %s -> %s", __FILE__, __LINE__, #call, hipGetErrorString(e_));        \
      return TCPXU_DEVICE_ERROR;                                                                     \
    }                                                                                                \
  } while (0)

#define TCPXU_TRY(call)                   \
  do {                                    \
    int rc_ = (call);                     \
    if (rc_ != TCPXU_SUCCESS) return rc_; \
  } while (0)

#endif  // TCPXU_HIP_COMMON_H_
