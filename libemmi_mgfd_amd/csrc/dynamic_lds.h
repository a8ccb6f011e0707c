// dynamic_lds.h -- kernels with more than the default 64 KiB of dynamic LDS.
#pragma once

#include <hip/hip_runtime.h>
#include <mutex>
#include <set>
#include <utility>

namespace emmi {

constexpr int CU_LDS = 160 * 1024;   // LDS of a CU

// allows the kernel at fn all of a CU's LDS on the current device; asked of the
// runtime once per kernel and device (a failure is asked again by the next call)
inline hipError_t allow_lds(const void* fn) {
  static std::mutex mu;
  static std::set<std::pair<const void*, int>> done;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(mu);
  if (done.count({fn, dev})) return hipSuccess;
  e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, CU_LDS);
  if (e == hipSuccess) done.insert({fn, dev});
  return e;
}

}  // namespace emmi
