// internal.h -- what the library's translation units share: the thread-local
// error string behind prh_last_error().
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

namespace prh_internal {
// record `msg` as the thread's last error; returns 1
int32_t error(const std::string& msg);
// 0, or record "what: <hip error>" and return 1
int32_t check(hipError_t e, const char* what);
}  // namespace prh_internal
