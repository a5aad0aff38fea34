// What the dense fp16 kernels share: their arguments, the numbering of tiles and
// slices, and the loads that write LDS directly.
#pragma once
#include <hip/hip_runtime.h>

#include "w4a16_common.hpp"

namespace w4a16 {

constexpr int kDnStageK = 64;    // k depth of a stage (two MFMA k steps); k is a multiple
constexpr int kDnOob = (int)0x80000000;
constexpr int kDnMaxSlices = 4;
constexpr int kDnCounterStride = 16;  // ints: a tile's slices meet in a cache line of their own

struct DenseArgs {
  const void* A;
  const void* B;
  void* C;
  int M, N, K;
  int tiles_m, tiles_n;
  int dp_tiles;  // tiles computed by one workgroup each
  // dense_small_kernel, in a launch of its own: the tiles after the first
  // dp_tiles, in ksplit slices each; with quarters, the plan's tiles are 256 x
  // 256 and computed as four tiles each
  int sk_tiles;
  int ksplit;
  int quarters;
  int* locks;        // one zeroed counter per cut tile, kDnCounterStride ints apart, zero again afterwards
  float* scratch;    // kPartBytes per slice
  int finish_polls;  // looks at a tile's other slices before leaving them a share
};

// Tiles are numbered panel by panel: a panel is kDnPanel column tiles wide
// (the last one narrower), and inside a panel the column tile runs fastest, or
// the row tile where there are fewer than kDnPanel of them.  A run of
// consecutive tile numbers then covers a compact block of C, so the workgroups
// that share an L2 read few distinct rows of A and B, and with few row tiles
// every row of B comes from memory into one L2 only (777 x 4352 x 10240: 91.5 us,
// with columns first 98.7).
constexpr int kDnPanel = 8;
__host__ __device__ __forceinline__ void dn_tile_coord(int t, int tiles_m, int tiles_n, int* tm,
                                                       int* tn) {
  const int per_panel = tiles_m * kDnPanel;
  const int p = t / per_panel;
  const int first = p * kDnPanel;
  const int width = tiles_n - first < kDnPanel ? tiles_n - first : kDnPanel;
  const int o = t - p * per_panel;
  if (tiles_m < kDnPanel) {
    *tn = first + o / tiles_m;
    *tm = o - (*tn - first) * tiles_m;
  } else {
    *tm = o / width;
    *tn = first + o - *tm * width;
  }
}

// (tile, slice) of a workgroup of a launch of slices: the slices of a tile are
// neighbours behind one L2, where they meet.  With the slices of one k range as
// neighbours instead, rows of B were shared by more tiles, but the sums passed
// between XCDs: 2226 x 768 x 1536 15.3 us, with this 12.9; 560 x 2560 x 2304 17.0
// and 15.0; four slices, 488 x 2048 x 1152 15.6 and 11.2; 350 x 2048 x 4096 17.9 and
// 15.0; quarters, 4096 x 4352 x 4096 118.0 and 118.2.
__host__ __device__ __forceinline__ void dn_slice_coord(int block, int tiles, int slices, int* tile,
                                                        int* slice) {
  const int work = xcd_work_index(block, tiles * slices);
  *tile = work / slices;
  *slice = work - *tile * slices;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t dn_rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}

// 16 bytes per lane from a buffer straight into LDS: lane l's bytes land at
// dst + 16*l (dst is wave-uniform).  The instruction's immediate offset stays
// zero: the hardware would add it to the LDS address as well.  (Device pass
// only; the host pass just needs the kernel's launch stub.)
__device__ __forceinline__ void dn_dma16(__amdgpu_buffer_rsrc_t rsrc, char* dst, int voffset,
                                         int soffset) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) void* lds_ptr;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)dst, 16, voffset, soffset, 0, 0);
#endif
}

// LDS reads of a main loop, outside the compiler's dependence tracking (it
// would wait for every load in flight before each of them)
template <int OFF>
__device__ __forceinline__ void dn_read16(unsigned at, i4& v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFF) : "memory");
#endif
}

// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding)
constexpr int dn_vmcnt(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }

__device__ __forceinline__ h4 dense_round(f4 v) {
  return (h4){(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
}

// One launch of a plan: `tiles` tiles of rows x cols in `slices` slices each, a
// workgroup of 64 * waves threads per slice
struct DnLaunch {
  int rows, cols, waves, tiles, slices;
};

// Tiles of f16_tiles.hip: rows x cols, in `slices` slices of the k range each; rows = 0
// where the plan's are the better ones.
struct DnTile {
  int rows, cols, slices;
};
// for a problem that `plan` alone would compute on a device of `cus` compute units; no
// more slices than that has
DnTile dn_tile(int m, int n, int k, int cus, const DnLaunch& plan);
bool dn_tile_exists(int rows, int cols, bool cut);
hipError_t configure_dense_tiles();
void launch_dense_tiles(DenseArgs a, const DnTile& t, hipStream_t stream);

}  // namespace w4a16
