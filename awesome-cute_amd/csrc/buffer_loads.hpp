// What the kernels' buffer instructions share: resources, loads that write LDS
// directly, LDS reads outside the compiler's tracking, and the wait for loads.
#pragma once
#include <hip/hip_runtime.h>

#include "w4a16_common.hpp"

namespace w4a16 {

constexpr int kOob = (int)0x80000000;  // offset past any buffer (sizes are < 2 GiB)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}

// the four words of a raw buffer resource: 48-bit base, stride 0, size in
// bytes, data format flags
__device__ __forceinline__ i4 rsrc_words(const void* p, unsigned bytes) {
  const unsigned long long a = (unsigned long long)p;
  return (i4){(int)(unsigned)a, (int)(unsigned)((a >> 32) & 0xffffu), (int)bytes, 0x00020000};
}

// 16 bytes per lane from a buffer straight into LDS: lane l's bytes land at
// dst + 16*l (dst is wave-uniform).  The instruction's immediate offset stays
// zero: the hardware would add it to the LDS address as well.  (Device pass
// only; the host pass just needs the kernel's launch stub.)  AUX 2: read once, not to
// stay in the caches.
template <int AUX = 0>
__device__ __forceinline__ void load_to_lds16(__amdgpu_buffer_rsrc_t rsrc, char* dst, int voffset,
                                              int soffset) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) void* lds_ptr;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)dst, 16, voffset, soffset, 0, AUX);
#endif
}

// LDS reads of a main loop, outside the compiler's dependence tracking (it
// would wait for every load in flight before each of them)
template <int OFF>
__device__ __forceinline__ void read_lds16(unsigned at, i4& v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFF) : "memory");
#endif
}

// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding)
constexpr int vmcnt(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }

}  // namespace w4a16
