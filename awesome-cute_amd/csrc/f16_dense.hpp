// What the dense fp16 kernels share: their arguments and the numbering of tiles and
// slices.
#pragma once
#include <hip/hip_runtime.h>

#include "buffer_loads.hpp"
#include "w4a16_common.hpp"

namespace w4a16 {

constexpr int kDnStageK = 64;    // k depth of a stage (two MFMA k steps); k is a multiple
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
