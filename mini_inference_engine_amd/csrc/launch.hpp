// What the launching code of several kernel files shares: more LDS than a kernel gets by default, the number of compute units,
// and the wait of kernels that count the loads they have on their way themselves.
#pragma once

#include "common.hpp"
#include <mutex>
#include <set>
#include <utility>

// wait until at most n vector memory loads of this wave are still on their way
#define MIE_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

// Ask for `bytes` of dynamic LDS, once a kernel and device; `what` begins the message of a refusal.
static inline int mie_allow_lds(const void* kernel, int bytes, const char* what) {
  static std::mutex lock;
  static std::set<std::pair<int, const void*>> done;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) MIE_FAIL("%s: no current device", what);
  std::lock_guard<std::mutex> g(lock);
  if (done.count({dev, kernel})) return 0;
  hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) MIE_FAIL("%s: %d bytes of LDS refused: %s", what, bytes, hipGetErrorString(e));
  done.insert({dev, kernel});
  return 0;
}

// of the current device (256 where that cannot be asked)
static inline int mie_compute_units() {
  static int units[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!units[dev]) {
    int n = 0;
    units[dev] = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
  }
  return units[dev];
}
