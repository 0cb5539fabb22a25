// march_launch.h -- host side of a march: one cooperative launch, in order with the
// other marches of its device.  Host code only (HIP runtime calls).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <mutex>

#include "internal.h"

namespace prh_internal {

// Marches of one process on one device run one after the other, whatever streams
// they are on: each waits for the event of the one before.  Two of them on the
// chip together could each hold CUs the other's barriers need.
constexpr int MAX_DEVICES = 64;
inline std::mutex g_order_mu;
inline hipEvent_t g_last_march[MAX_DEVICES] = {};

// A march belongs to its stream's device: the event that orders it and the dynamic
// LDS limit of its kernel are that device's, whichever one the caller has current.
struct StreamDevice {
  int id = -1, before = -1;
  hipError_t error;
  explicit StreamDevice(hipStream_t s) {
    error = hipStreamGetDevice(s, &id);
    if (error == hipSuccess) error = hipGetDevice(&before);
    if (error == hipSuccess && id != before) error = hipSetDevice(id);
  }
  ~StreamDevice() {
    if (before >= 0 && id != before) (void)hipSetDevice(before);
  }
  StreamDevice(const StreamDevice&) = delete;
  StreamDevice& operator=(const StreamDevice&) = delete;
};

struct MarchLaunch {
  const void* reset;   // one workgroup, argument sync: clears the sync words
  const void* march;   // the cooperative kernel
  const void* behind;  // voids an aborted march's results (same arguments)
  unsigned blocks, threads;
  size_t lds;
  uint32_t* sync;
  void* args;
};

// status: nothing was launched, the stage kernels can run instead
constexpr int32_t NOT_LAUNCHABLE = 2;

// Whether the device can hold the whole grid at once; asked before the launch, so that
// stepping aside leaves no runtime error behind for the next call to report.
inline hipError_t march_fits(const MarchLaunch& m, int dev, bool& fits) {
  int coop = 0, lds = 0, cus = 0, per_cu = 0;
  fits = false;
  hipError_t e = hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev);
  if (e == hipSuccess)
    e = hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess || !coop || m.lds > (size_t)lds) return e;
  e = hipFuncSetAttribute(m.march, hipFuncAttributeMaxDynamicSharedMemorySize, (int)m.lds);
  if (e == hipSuccess)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, m.march, (int)m.threads, m.lds);
  fits = e == hipSuccess && (int64_t)per_cu * cus >= m.blocks;
  return e;
}

inline int32_t launch_march(const MarchLaunch& m, hipStream_t s) {
  const StreamDevice dev(s);
  if (dev.error != hipSuccess) return check(dev.error, "team march: device of the stream");
  if (dev.id < 0 || dev.id >= MAX_DEVICES) return error("team march: no device in [0, 64)");
  bool fits;
  hipError_t e = march_fits(m, dev.id, fits);
  if (e != hipSuccess) return check(e, "team march: what the device holds");
  if (!fits) {
    error("team march: the device cannot hold the grid");
    return NOT_LAUNCHABLE;
  }
  std::lock_guard<std::mutex> lock(g_order_mu);
  hipEvent_t& last = g_last_march[dev.id];
  e = last ? hipStreamWaitEvent(s, last, 0)
           : hipEventCreateWithFlags(&last, hipEventDisableTiming);
  if (e != hipSuccess) return check(e, "team march: order");
  uint32_t* sync = m.sync;
  void* reset_args[] = {&sync};
  void* args[] = {m.args};
  e = hipLaunchKernel(m.reset, dim3(1), dim3(1024), reset_args, 0, s);
  if (e == hipSuccess)
    e = hipLaunchCooperativeKernel(m.march, dim3(m.blocks), dim3(m.threads), args,
                                   (unsigned)m.lds, s);
  if (e == hipSuccess) e = hipLaunchKernel(m.behind, dim3(256), dim3(256), args, 0, s);
  if (e == hipSuccess) e = hipEventRecord(last, s);
  const int32_t rc = check(e, "team march launch");
  if (e != hipErrorCooperativeLaunchTooLarge && e != hipErrorNotSupported) return rc;
  (void)hipGetLastError();  // refused after all: no error is left for the stage kernels' checks
  return NOT_LAUNCHABLE;
}

}  // namespace prh_internal
