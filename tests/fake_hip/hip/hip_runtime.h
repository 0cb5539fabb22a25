// The HIP runtime calls of csrc/march_launch.h as a host-only model with two devices:
// what a call needs of streams, events and the current device is checked as the
// runtime does, and every call is written to a log.
#pragma once

#include <cstddef>
#include <map>
#include <string>
#include <utility>

enum hipError_t {
  hipSuccess = 0,
  hipErrorInvalidValue = 1,
  hipErrorInvalidHandle = 400,
  hipErrorCooperativeLaunchTooLarge = 720,
  hipErrorNotSupported = 801
};
struct FakeStream {
  int device;
};
struct FakeEvent {
  int device;
  bool recorded;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;
struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
enum { hipFuncAttributeMaxDynamicSharedMemorySize = 8, hipEventDisableTiming = 2 };
enum hipDeviceAttribute_t {
  hipDeviceAttributeCooperativeLaunch,
  hipDeviceAttributeMaxSharedMemoryPerBlock,
  hipDeviceAttributeMultiprocessorCount
};

namespace fake {
inline int current = 0;
inline hipError_t last = hipSuccess;  // the latest error, until it is read
inline std::string log;
inline std::map<std::pair<int, const void*>, int> lds;  // limit set per device and kernel
inline unsigned max_blocks = 256;  // a cooperative launch may have
inline int lds_max = 163840, per_cu = 1, coop = 1;  // what the device says of itself
inline int device_of(hipStream_t s) { return s ? s->device : current; }
inline hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}
inline void note(const char* what, int device) {
  log += std::string(what) + std::to_string(device) + " ";
}
}  // namespace fake

inline hipError_t hipGetDevice(int* d) {
  *d = fake::current;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  if (d < 0 || d > 1) return fake::ret(hipErrorInvalidValue);
  fake::current = d;
  return hipSuccess;
}
inline hipError_t hipStreamGetDevice(hipStream_t s, int* d) {
  *d = fake::device_of(s);
  return hipSuccess;
}
inline hipError_t hipGetLastError() {
  const hipError_t e = fake::last;
  fake::last = hipSuccess;
  return e;
}
inline hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeCooperativeLaunch         ? fake::coop
       : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? fake::lds_max
                                                        : 256;
  return hipSuccess;
}
inline hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = fake::per_cu;
  return hipSuccess;
}
inline hipError_t hipFuncSetAttribute(const void* fn, int, int bytes) {
  if (bytes > fake::lds_max) return fake::ret(hipErrorInvalidValue);
  fake::lds[{fake::current, fn}] = bytes;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new FakeEvent{fake::current, false};
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->device != fake::device_of(s)) return fake::ret(hipErrorInvalidHandle);
  e->recorded = true;
  fake::note("record", e->device);
  return hipSuccess;
}
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  fake::note("wait", e->device);
  return hipSuccess;
}
inline hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t s) {
  fake::note("kernel", fake::device_of(s));
  return hipSuccess;
}
inline hipError_t hipLaunchCooperativeKernel(const void* fn, dim3 g, dim3, void**, unsigned lds,
                                             hipStream_t s) {
  const int d = fake::device_of(s);
  if (lds > 65536 && fake::lds[{d, fn}] < (int)lds) return fake::ret(hipErrorInvalidValue);
  if (g.x > fake::max_blocks) return fake::ret(hipErrorCooperativeLaunchTooLarge);
  fake::note("march", d);
  return hipSuccess;
}
