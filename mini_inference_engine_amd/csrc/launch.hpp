// What the launching code of several kernel files shares: more LDS than a kernel gets by default, the number of compute units,
// and the wait of kernels that count the loads they have on their way themselves.
#pragma once

#include "common.hpp"
#include <mutex>
#include <set>
#include <utility>

// wait until at most n vector memory loads of this wave are still on their way
#define MIE_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

// 16 bytes a lane from base + offset into the LDS at byte `at` + 16 lane.  The compiler does not see that memory is on its
// way: the waits are the kernel's own (MIE_VMCNT and a barrier before a stage is read).  m0 is an output, so that the
// compiler keeps nothing of its own there; as an input operand it costs the loop its order of moves and loads (2,048 rows of
// [11264, 2048] 90.1 -> 93.0 us).
__device__ __forceinline__ void mie_load_to_lds(const void* base, uint32_t offset, uint32_t at) {
  uint32_t written;
  asm volatile(
    "s_mov_b32 m0, %1\n\t"
    "s_nop 0\n\t"
    "global_load_lds_dwordx4 %2, %3"
    : "={m0}"(written)
    : "s"(at), "v"(offset), "s"(base)
    : "memory");
}

// the same with the hint of loads whose lines nobody reads again: weights that one workgroup takes
__device__ __forceinline__ void mie_load_to_lds_nt(const void* base, uint32_t offset, uint32_t at) {
  uint32_t written;
  asm volatile(
    "s_mov_b32 m0, %1\n\t"
    "s_nop 0\n\t"
    "global_load_lds_dwordx4 %2, %3 nt"
    : "={m0}"(written)
    : "s"(at), "v"(offset), "s"(base)
    : "memory");
}

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
