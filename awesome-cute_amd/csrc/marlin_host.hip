// Host launcher and C ABI of the gfx950 W4A16 Marlin GEMM.
//
// Mirrors the host side of the reference path: the argument contract and
// shape checks of marlin_cute (marlin_cute_kernel.cu:28-115) and the checks
// of the tensor binding mul (marlin_gemm.cpp:19-56).  Kernel choice, grid and
// partition are this library's own.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <mutex>
#include <vector>

#include "../../include/marlin_amd.h"
#include "../../include/marlin_amd_tools.h"
#include "scratch_pool.hpp"
#include "w4a16_common.hpp"

// Scratch for partial sums and tile counters that marlin_gemm_static uses in
// place of the pool's allocations: a fixed array in device memory, one copy per
// GPU, addressed through the pointer hipGetSymbolAddress returns for the
// current device (the name itself is not a device address in host code).
constexpr size_t kStaticPartialBytes = (size_t)32 << 20;
constexpr size_t kStaticScratchBytes = w4a16::kCounterBytes + kStaticPartialBytes;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace w4a16 {
hipError_t& last_launch_error() {
  thread_local hipError_t e = hipSuccess;
  return e;
}
}  // namespace w4a16

namespace {

using namespace w4a16;

constexpr int kMaxStreamGrid = 1024;  // workgroups of the streaming kernel
constexpr int kMaxDevices = 16;

thread_local char g_last_error[256] = "";

void set_error(hipError_t e, const char* what) {
  snprintf(g_last_error, sizeof(g_last_error), "%s: %s", what, hipGetErrorString(e));
}

struct DeviceState {
  int cus = 0;
  bool configured = false;          // kernels' LDS limits raised on this device
  unsigned char* static_scratch = nullptr;  // this device's copy of `scratch`
};
std::mutex g_mu;
DeviceState g_dev[kMaxDevices];

// What the planner may assume about the partial-sum buffer: the pool grows up
// to this much for one call; the fixed array of marlin_gemm_static is smaller.
constexpr size_t kPoolPartialLimit = (size_t)64 << 20;

// With `dev` current: raise the dynamic-LDS limit of the kernels that need it.
bool configure_device(int dev) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_dev[dev].configured) return true;
  if (configure_stream_kernels() != 0 || configure_prefill_kernels() != 0 ||
      configure_prefill_wide_kernels() != 0 || configure_strip_kernels() != 0 ||
      configure_rows_kernels() != 0 || configure_rows_wide_kernels() != 0) {
    set_error(hipGetLastError(), "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
    return false;
  }
  g_dev[dev].configured = true;
  return true;
}

int device_cus(int dev) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_dev[dev].cus == 0) {
    int cus = 0;
    hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) {
      set_error(e, "hipDeviceGetAttribute");
      return -1;
    }
    g_dev[dev].cus = cus;
  }
  return g_dev[dev].cus;
}

// Shape checks in the order the reference performs them
// (marlin_cute_kernel.cu:39-60, 95-107).
int check_shape(int m, int n, int k, int groupsize, int& thread_k, int& thread_n) {
  if (thread_k == -1 || thread_n == -1) {
    if (m <= 16) {
      thread_k = 128;
      thread_n = 128;
    } else {
      thread_k = 64;
      thread_n = 256;
    }
  }
  if (thread_k <= 0 || thread_n <= 0) return MARLIN_ERR_PROB_SHAPE;
  if (groupsize == 0 || groupsize < -1) return MARLIN_ERR_KERN_SHAPE;
  const int group_blocks = groupsize == -1 ? -1 : groupsize / 16;
  if (group_blocks == 0) return MARLIN_ERR_KERN_SHAPE;
  if (m < 0 || n < 0 || k < 0) return MARLIN_ERR_PROB_SHAPE;
  if (n % thread_n != 0 || k % thread_k != 0 || (group_blocks != -1 && k % group_blocks != 0))
    return MARLIN_ERR_PROB_SHAPE;
  if (m == 0 || n == 0 || k == 0) return MARLIN_OK;
  // kernel table: tiles (128 k x 128 n) for one 16-row block, (64 k x 256 n)
  // for one to four; group size 128 or per-channel
  if (groupsize != -1 && groupsize != 128) return MARLIN_ERR_KERN_SHAPE;
  const bool small = thread_k == 128 && thread_n == 128;
  const bool wide = thread_k == 64 && thread_n == 256;
  if (!small && !wide) return MARLIN_ERR_KERN_SHAPE;
  if (small && m > 16) return MARLIN_ERR_KERN_SHAPE;
  if (groupsize == 128 && k % 128 != 0) return MARLIN_ERR_PROB_SHAPE;
  return MARLIN_OK;
}

struct Plan {
  int kernel;  // 1 streaming, 2 prefill, 3 column strips
  int grid;
  StreamPlan sp;
  int launches;
  int ksplit;            // prefill: slices of the k range per tile
  int tile_rows;         // prefill: rows of C per workgroup
  size_t partial_bytes;  // fp32 partial sums the launch exchanges through scratch (0: none)
  int row_parts;         // streaming, one-tile form: parts the rows are cut into (1: uncut)
  int part_rows;         // rows of a part (the last one has the rest)
  int strips;            // column-strip kernel: 16-column strips per workgroup (else 0)
};

constexpr int kStreamMaxRows = 64;
constexpr int kSliceCounterStride = 16;  // ints: a prefill tile's slices meet in a cache line of their own

// Overrides of the planner for the calling thread (tests and tools; see
// marlin_amd_force_*): which kernel (0 = by cost, 1 = streaming in chunks of
// 64 rows, 2 = prefill, 3 = column strips, 4 = by cost without the column
// strips), slices of the k range per prefill tile (0 = by cost),
// rows of C per prefill workgroup (0 = by cost, 64 to 128 in steps of 16).
struct Force {
  int kernel = 0, k_slices = 0, tile_rows = 0;
  int row_halves = 0;  // streaming kernel: 0 = by cost, 1 = never cut the rows, 2 = cut them where possible
  int strips = 0;      // column-strip kernel: 0 = by cost, or 1 to 4 strips per workgroup
  int rows_strips = 0, rows_blocks = 0;  // rows of a strip set in one workgroup: 0 = by cost, strips -1 = never
  int finish_polls = -1;  // looks at the other slices of a tile before leaving; -1 = kFinishPolls
  bool any() const {
    return kernel != 0 || k_slices != 0 || tile_rows != 0 || row_halves != 0 || strips != 0 ||
           rows_strips != 0 || finish_polls >= 0;
  }
};
thread_local Force t_force;

// What a plan is made for: the device's compute units, the room for partial
// sums, and the thread's overrides.
struct PlanCtx {
  int cus;
  size_t partial_limit;
  Force force;
  bool grouped;       // scales per group of 128, or one per column
  int counters = 16;  // ints of the workspace per column tile: min(max_par, 16)
};

// Cost in us of the prefill kernels with `tiles` tiles of tile_rows rows cut
// into s slices, linear in what they do: a launch, a round of workgroups, a
// 64-deep stage of each k half of a workgroup (dearer the fuller the chip: the
// board's power), and with slices their meeting, dearer with their number and
// with the traffic of a full chip.  R is the row blocks of a tile of the
// four-wave kernel.  Fitted to launches on MI355X, by themselves with group scales
// (2700, M = 65 ... 2100 on eleven (N, K) from 1024 x 1024 to 28672 x 8192, every
// tile height and slice count; 4 % rms for 64 rows, 5 % for the others) and with
// one scale per column (32000 over 1300 problems, M = 33 ... 8192; 5 and 6 %),
// whose weights are unpacked without a scale to multiply: a stage of a 64-row
// tile takes 0.83 of the time, one of a 128-row tile 0.92.  By the first fit for
// both, one problem in thirty with a scale per column was given slices or rows that
// took 5 to 20 % longer than others (M = 313, N = 4096, K = 9728: five slices of 112
// rows 33.1 us, three of 64 29.2).
double prefill_cost_slices(int tiles, int tile_rows, int k, const PlanCtx& cx, int s) {
  // more workgroups than CUs run in rounds, the last of which is faster the
  // emptier it is: half way between whole rounds and the plain ratio fits
  const double ratio = (double)tiles * s / cx.cus;
  const int whole = ceil_div(tiles * s, cx.cus);
  const double rounds = ratio <= 1.0 ? 1.0 : 0.5 * (whole + ratio);
  const double fill = ratio < 1.0 ? ratio : 1.0;
  const int depth = ceil_div(ceil_div(ceil_div(k, 64), s), 2);
  const double stages = rounds * depth;
  const double R = tile_rows / 16.0;
  if (cx.grouped && tile_rows == 64)
    return -2.24 + 7.07 * rounds + (0.753 + 0.256 * fill) * stages +
           (s > 1 ? 0.86 + 0.61 * s + 1.90 * fill * rounds : 0.0);
  if (cx.grouped)
    return 5.16 - 1.97 * R + (2.63 * R - 2.42) * rounds +
           (0.519 + (0.0586 + 0.0419 * fill) * R) * stages +
           (s > 1 ? 2.12 + 0.302 * s + 0.625 * fill * rounds * R : 0.0);
  const double late = ratio <= 1.0 ? 0.0 : (double)whole * depth;
  if (tile_rows == 64)
    return 2.34 + 3.22 * rounds + (0.656 + 0.116 * fill) * stages + 0.121 * late +
           (s > 1 ? 0.508 + 0.629 * s + 2.16 * fill * rounds : 0.0);
  return 3.92 - 0.318 * R + (0.960 * R - 0.802) * rounds +
         (0.314 + (0.0704 + 0.0289 * fill) * R) * stages + 0.173 * late +
         (s > 1 ? 3.33 + 0.290 * s + 0.501 * fill * rounds * R : 0.0);
}

// Whether a tile height is cut into s slices at all.  With 64 rows no more than
// six (eight gain nothing where the streaming kernel does not win anyway: M =
// 100, N = 4096, K = 11008 24.1 us with six, 25.3 with eight).  Three row
// blocks per wave finish in six pieces, which only 2, 3 and 6 slices share
// evenly (80 rows, M = 150, N = 4096, K = 11008: four slices 31.0 us, five
// 28.6, six 26.4, seven 28.0, eight 27.8); eight pieces are less particular.
bool slices_share(int tile_rows, int s) {
  if (tile_rows == 64) return s <= 6;
  return tile_rows > 96 || 6 % s == 0;
}

// Slices of the k range per tile: the cheapest count among those that keep
// the launch within one workgroup per CU, slices at least 256 deep (two
// 64-deep stages for each half of the workgroup), and the partial sums and
// tile counters within the scratch.  Up to eight.
int prefill_k_slices(int tiles, int tile_rows, int k, const PlanCtx& cx) {
  int most = k / 256;
  if (most > kMaxSlices) most = kMaxSlices;
  while (most > 1 && (size_t)tiles * most * ceil_div(tile_rows, 32) * 32 * 256 * 4 > cx.partial_limit)
    --most;
  if (most < 1 || tiles > kMaxCounters / kSliceCounterStride) return 1;
  if (cx.force.k_slices > 0) return cx.force.k_slices < most ? cx.force.k_slices : most;
  if (most > cx.cus / tiles) most = cx.cus / tiles;
  int best = 1;
  double best_cost = prefill_cost_slices(tiles, tile_rows, k, cx, 1);
  for (int s = 2; s <= most; s++) {
    if (!slices_share(tile_rows, s)) continue;
    const double c = prefill_cost_slices(tiles, tile_rows, k, cx, s);
    if (c < best_cost) {
      best = s;
      best_cost = c;
    }
  }
  return best;
}

double prefill_cost_rows(int m, int n, int k, const PlanCtx& cx, int tile_rows) {
  const int tiles = ceil_div(m, tile_rows) * (n / 256);
  return prefill_cost_slices(tiles, tile_rows, k, cx,
                             prefill_k_slices(tiles, tile_rows, k, cx));
}

// Rows of C per prefill workgroup: the cheapest of 64 (eight waves) and 80 to
// 128 in steps of 16 (four).  Heights other than 64 and 128 are there for row
// counts that 64-row tiles would pad -- M = 150, N = 12288, K = 4096: 31.6 us
// with 64 rows, 31.7 with 128, 26.0 with 80; M = 300, N = K = 8192 59.1, 51.2
// and 45.4; M = 203, N = 5120, K = 13568 46.8, 42.6 and 40.1 with 112; M = 300,
// N = 28672, K = 8192 189, 172 and 142 -- and have to be ahead by 2 %, about what
// the fit is worth.  Over 1660 problems that leaves 12 (14 with one scale per
// column) that take 2 to 11 % longer than with 64 or 128 rows, 17 (54) without it
// and with one fit for both; all together take 0.96 of the time.  (Where M is a
// multiple of 64 they are not tried.)
int prefill_tile_rows(int m, int n, int k, const PlanCtx& cx) {
  if (cx.force.tile_rows != 0) return cx.force.tile_rows;
  if (m <= 64) return 64;
  int best = 64;
  double best_cost = prefill_cost_rows(m, n, k, cx, 64);
  for (int rows = m % 64 == 0 ? 128 : 80; rows <= 128; rows += 16) {
    const double c = prefill_cost_rows(m, n, k, cx, rows) * (rows == 128 ? 1.0 : 1.02);
    if (c < best_cost) {
      best = rows;
      best_cost = c;
    }
  }
  return best;
}

double prefill_cost(int m, int n, int k, const PlanCtx& cx) {
  return prefill_cost_rows(m, n, k, cx, prefill_tile_rows(m, n, k, cx));
}

// The streaming kernel's split of the granule sequence over the compute units
// for `mb` row blocks.  Measured on MI355X: a split that keeps every workgroup
// inside one column tile (or gives it whole tiles) costs about 0.1 us x row
// blocks per granule of the longest workgroup; a split that leaves workgroups
// straddling tile boundaries is several us slower (a second exchange per
// workgroup, and workgroups that read different weight rows at the same
// time), about 1 + 2.5 x row blocks us.  Candidates: every tile cut into c
// nearly equal runs (c tiles' worth of workgroups <= CUs), whole tiles per
// workgroup, and the evenly balanced uniform split.
struct StreamSplit {
  int gpb;        // granules of the longest workgroup
  int wpt;        // workgroups per column tile, or 0 for the uniform form
  bool straddle;  // workgroups cross tile boundaries
};
// The last arrival of a tile fetches its sharers eight at a time: beyond 8
// every sharer costs (M = 16, N = 2048, K = 4096: 8 runs per tile 6.1 us, 16
// 6.7, 32 10.7; N = 1024, K = 8192: 8 7.9, 16 7.1, 32 8.9)
double sharer_cost(int c) { return c <= 8 ? 0.0 : c <= 16 ? 0.1 * (c - 8) : 0.8 + 0.25 * (c - 16); }

StreamSplit choose_stream_split(int mb, int n, int k, int cus) {
  const int NT = n / kTileN;
  const int KG = k / kGranuleK;
  const int total = NT * KG;
  if (cus > kMaxStreamGrid) cus = kMaxStreamGrid;  // the grid the kernel's slots allow
  const double per_granule = 0.1 * mb, straddle = 1.0 + 2.5 * mb;
  StreamSplit sp;
  sp.gpb = ceil_div(total, cus);
  sp.wpt = 0;
  sp.straddle = !(sp.gpb % KG == 0 || KG % sp.gpb == 0);
  auto sharers = sharer_cost;
  double best_cost = per_granule * sp.gpb + (sp.straddle ? straddle : 0.0) +
                     sharers(ceil_div(KG, sp.gpb));
  for (int c = 1; c <= KG && NT * c <= cus; c++) {
    const int g = ceil_div(KG, c);
    const double cost = per_granule * g + sharers(c);
    if (cost < best_cost + 1e-9) {  // on a tie the one-tile form: its kernel is leaner
      sp.gpb = g;
      sp.wpt = c;
      sp.straddle = false;
      best_cost = cost;
    }
  }
  for (int mult = 2; mult * KG <= total; mult++) {
    const int g = mult * KG;
    if (ceil_div(total, g) > cus) continue;  // more workgroups than CUs never paid off
    const double cost = per_granule * g;
    if (cost < best_cost - 1e-9) {
      sp.gpb = g;
      sp.wpt = 0;
      sp.straddle = false;
      best_cost = cost;
    }
  }
  return sp;
}

// What cutting the rows of a streaming launch in two saves (us; negative: a
// loss), fitted on MI355X over N = 2048...11008, K = 4096...13824, 17 to 64
// rows.  The halves have half the row blocks to sum, store and read back and
// half the sharers per tile, which is worth S; their runs are twice as long,
// and a granule of one or two row blocks costs more than half a granule of two
// to four, which costs p per granule of the uncut run.  S jumps where the last
// arrival of the uncut launch would fetch its sharers in more than one round
// (more than 8).  E.g. M = 64, N = K = 4096 (8 sharers, 8 granules): 12.9 ->
// 10.2 us; N = 2048: 14.9 -> 8.5; 8192 x 8192 (4 sharers, 32 granules): 20.0
// -> 19.5; M = 48 there 17.1 -> 19.1 (not cut).
double halves_gain(int rows, int wpt, int gpb) {
  const int mb = ceil_div(rows, 16);
  const bool rounds = wpt > 8;
  const double p = 0.06;
  double s;
  if (mb <= 2)
    s = rounds ? 2.8 : 1.0 + 0.045 * (rows - 16);
  else if (mb == 3)
    s = rounds ? 4.0 : 1.0 + 0.027 * (rows - 33);
  else
    s = rounds ? 6.5 : 3.2;
  return s - p * gpb;
}

// Fitted time (us) of the streaming kernel with uncut rows: a pass over 49-64
// rows takes 11.3 + 0.28 per granule of the longest workgroup (N=K=4096: 8
// granules, 12.9; N=8192, K=4096: 16, 15.5; N=4096, K=11008: 22, 18.0;
// N=11008, K=4096 or 8192^2: 32, 18.5-20; N=28672, K=8192: 128, 46), fewer
// rows a share of that, up to 16 rows 4.9 + 0.17 per granule (1.4 less where
// no tile is shared: N=28672, K=8192, 128 granules, 23 us); every launch
// after the first waits a microsecond for the one before (65 rows at N=4096,
// K=11008: 18.0 + 9.0 alone, 27.0 in a row).
double stream_cost(int m, int n, int k, int cus) {
  const StreamSplit s4 = choose_stream_split(4, n, k, cus);
  const double full = 11.3 + 0.28 * s4.gpb + (s4.straddle ? 11.0 : 0.0);
  const int tail = m % kStreamMaxRows;
  double t = (m / kStreamMaxRows) * full;
  if (tail > 16) {
    t += full * (tail > 48 ? 1.0 : tail > 32 ? 0.9 : 0.65);
  } else if (tail > 0) {
    const StreamSplit s1 = choose_stream_split(1, n, k, cus);
    // (refitted over M = 1, 4, 8, 16 on N = 256...28672, K = 512...11008, 6 %
    // rms: a workgroup that shares its tiles with no other exchanges nothing)
    const int sharers = s1.wpt > 0 ? s1.wpt : ceil_div(k / kGranuleK, s1.gpb);
    t += 4.94 + 0.167 * s1.gpb + (tail > 8 ? 0.23 : 0.0) + (s1.straddle ? 3.5 : 0.0) +
         (sharers == 1 && !s1.straddle ? -1.39 : sharer_cost(sharers));
  }
  return t + 1.0 * (ceil_div(m, kStreamMaxRows) - 1);
}

// More than 64 rows in one streaming launch: the rows cut into parts of 32,
// every (tile, part) a problem of its own for wpt workgroups.  Possible while
// there is a CU per (tile, part) and a counter per part; costs what a 32-row
// launch of that split costs (0.65 of the fit above; measured 12.6 us against
// 13.2 for M = 128 at N = K = 4096, 22.9 / 23.0 at K = 11008, 17.1 / 17.0 for
// M = 256 with one workgroup per tile and part).  Sets wpt
// and the granules per run; returns the cost in us, or a negative number where
// it cannot be done.
double stream_parts_cost(int m, int n, int k, const PlanCtx& cx, int* parts, int* wpt, int* gpb) {
  const int NT = n / kTileN, KG = k / kGranuleK;
  const int P = ceil_div(m, 32);
  if (m <= kStreamMaxRows || P > cx.counters || NT * P > cx.cus || cx.force.row_halves == 1)
    return -1.0;
  int w = cx.cus / (NT * P);
  if (w > KG) w = KG;
  // more than 8 sharers would be fetched in two rounds by the last arrival
  if (w > 8) w = 8;
  *parts = P;
  *wpt = w;
  *gpb = ceil_div(KG, w);
  // (a launch that exchanges nothing saves the 2 us the fit holds for that)
  return 0.65 * (11.3 + 0.28 * *gpb) - (w == 1 ? 2.0 : 0.0);
}

// 9 to 16 rows, one launch, by kind of scales: a launch that shares its tiles and one that does
// not, the granules of the longest workgroup, the weights' way from memory, runs that straddle
// tiles, sharers beyond eight.  1490 launches over N = 256 ... 28672, K = 512 ... 16384, 4 % rms.
// (By the fit above, without the weights and of group scales alone, one scale per column read 0.88
// of it where a tile has one workgroup and 1.05 with nine and more: 15 x 18176 x 4608 took 14.5 us
// as strips, 12.3 streaming, 14 x 2048 x 5504 7.0 streaming, 6.3 as strips.)
double stream_cost_few(int n, int k, const PlanCtx& cx) {
  const StreamSplit s = choose_stream_split(1, n, k, cx.cus);
  const int sharers = s.wpt > 0 ? s.wpt : ceil_div(k / kGranuleK, s.gpb);
  const bool alone = sharers == 1 && !s.straddle;
  const int beyond = sharers > 8 ? sharers - 8 : 0;
  const double MB = 0.5e-6 * n * k;
  if (cx.grouped)
    return (alone ? 3.77 : 5.08) + 0.108 * s.gpb + 0.073 * MB + (s.straddle ? 4.5 : 0.0) + 0.24 * beyond;
  return (alone ? 3.87 : 5.24) + 0.074 * s.gpb + 0.075 * MB + (s.straddle ? 4.4 : 0.0) + 0.24 * beyond;
}

// The streaming kernel's cost as make_plan would launch it: with the rows cut
// in two or into parts of 32 where that is cheaper.
double stream_cost_as_planned(int m, int n, int k, const PlanCtx& cx) {
  if (m > 8 && m <= 16) return stream_cost_few(n, k, cx);
  double stream = stream_cost(m, n, k, cx.cus);
  if (m <= kStreamMaxRows && cx.force.row_halves != 1 && cx.counters >= 2) {
    // what the launch gains where make_plan cuts its rows in two
    const StreamSplit split = choose_stream_split(ceil_div(m, 16), n, k, cx.cus);
    const int half = 16 * ceil_div(ceil_div(m, 2), 16);
    const StreamSplit hs = choose_stream_split(half / 16, 2 * n, k, cx.cus);
    const double gain = split.wpt >= 2 && hs.wpt >= 1 && half < m
                            ? halves_gain(m, 2 * hs.wpt, ceil_div(k / kGranuleK, 2 * hs.wpt))
                            : 0.0;
    if (gain > 0.25) {
      // (the halves take no less than a launch of half the rows over twice the
      // tiles: the gain was fitted where the uncut launch fetches its sharers
      // in rounds, which the fit of the uncut launch does not hold -- M = 64,
      // N = 2048, K = 4096: 12.1 - 6.3 by the fits, 8.7 us measured, 8.1 by this)
      const double alone = stream_cost(half, 2 * n, k, cx.cus);
      stream = stream - gain > alone ? stream - gain : alone;
    }
    // 17 to 64 rows over short, wide weights: tiles of at most 16 granules that
    // two to four workgroups share finish in three quarters of the fit's time
    // (K = 512 and 1024 at N = 4096...28672: 0.6 to 0.9 of it; N <= 2048, more
    // sharers per tile: 1.05 to 1.4)
    if (m > 16 && k < 2048 && n >= 4096) stream *= 0.75;
  }
  int parts, wpt, gpb;
  const double cut = stream_parts_cost(m, n, k, cx, &parts, &wpt, &gpb);
  if (cut > 0.0 && cut < stream) stream = cut;
  return stream;
}

bool prefer_prefill(int m, int n, int k, const PlanCtx& cx) {
  // no measurement favours 64-row prefill tiles below four row blocks
  if (m <= 48) return false;
  // ... nor, up to 64 rows, over weights that are neither wide nor deep: 56 and
  // 64 rows at N = 256...11008 with K = 512...4096 stream in 0.6 to 0.95 of
  // the prefill kernel's time (N = 28672: 1.07 to 1.1 at every K; N = 11008:
  // 1.1 at K = 8192, 1.5 at 11008), which the two fits, 15 % apart there in
  // opposite directions, do not resolve
  if (m <= kStreamMaxRows && n < 16384 && k < 8192) return false;
  // (the streaming kernel's fit is that of group scales; one scale per column
  // takes 0.96 of the time, and the fit is 5 % high where this is decided: M = 107,
  // N = 8192, K = 4096 15.5 us streaming, 16.5 in four slices of 64 rows, by the fits
  // 17.0 and 16.4)
  return prefill_cost(m, n, k, cx) <= stream_cost_as_planned(m, n, k, cx) * (cx.grouped ? 1.0 : 0.9);
}

// Fitted time (us) of the rows kernel (w4a16_rows.hip, w4a16_rows_wide.hip) with more than 16
// rows, also where it computes column strips in parts: a launch, the meeting of the waves' sums,
// the activations and weights a workgroup takes in and what it computes, dearer the fuller the
// chip, much the same again for workgroups beyond one per compute unit (by the rounds they make,
// and half way between these and their share of one), the weights' way from memory, and by how much
// the longest of the eight waves, and of the four SIMDs, is longer than the others where k does not
// divide evenly (ten groups: two for two of the waves, one for six).  And where the rows that an
// XCD's workgroups read outgrow its L2 -- an eighth of the strip sets each, with fewer than eight
// an eighth of (set, row part) pairs -- 0.4 us per MB beyond 3.5.  17600 launches over 3211
// problems, M = 17 ... 1500, N = 512 ... 28672, K = 640 ... 13824, 5 % rms.  The factors are those
// of the pairs, with group scales and without.
struct RowsPair {
  int strips, blocks;
  double by[2];
};
constexpr RowsPair kRowsPairs[] = {
    {1, 1, {1.060, 1.103}}, {2, 1, {0.999, 1.003}}, {3, 1, {1.045, 1.053}}, {2, 2, {1.000, 1.000}},
    {3, 2, {1.000, 0.993}}, {4, 2, {0.963, 0.927}}, {6, 2, {1.014, 0.952}}, {2, 3, {1.010, 0.976}},
    {3, 3, {0.982, 0.957}}, {4, 3, {1.008, 0.951}}, {5, 3, {1.036, 0.989}}, {6, 3, {1.037, 0.963}},
    {4, 4, {1.010, 1.000}}, {5, 4, {1.046, 1.008}}, {6, 4, {1.020, 0.950}}, {8, 2, {0.989, 0.940}},
    {8, 3, {0.999, 0.949}}, {8, 4, {1.004, 0.946}}, {4, 1, {1.016, 1.007}},
};
const RowsPair& rows_pair(int strips, int blocks) {
  const RowsPair* p = kRowsPairs;
  while (p->strips != strips || p->blocks != blocks) p++;  // (a pair of the table)
  return *p;
}
double rows_cost(int m, int n, int k, const RowsPair& p, const PlanCtx& cx) {
  const int sets = ceil_div(n / 16, p.strips);
  const int wgs = sets * ceil_div(m, 16 * p.blocks);
  const double r = (double)wgs / cx.cus;
  const double fill = r < 1.0 ? r : 1.0;
  const double more = r > 1.0 ? 0.5 * (ceil_div(wgs, cx.cus) + r) - 1.0 : 0.0;
  const int whole = ceil_div(wgs, cx.cus) - 1;
  const double K = k / 1000.0, b = p.blocks, s = p.strips, sums = b * s;
  const double memory = 0.5e-7 * n * k;
  const double out = 2e-6 * m * k * (sets < 8 ? sets / 8.0 : 1.0) - 3.5;
  const double beyond = out > 0.0 ? out : 0.0;
  // (the kernel deals out whole groups where there are more than four)
  const int unit = cx.grouped && k > 512 ? 128 : 64;
  const double wave = 8e-3 * unit * ceil_div(k / unit, 8) - K, simd = 4e-3 * unit * ceil_div(k / unit, 4) - K;
  double by = p.by[cx.grouped ? 0 : 1];
  // (six and eight strips with all rows in one workgroup take less)
  if (p.strips >= 6 && wgs == sets && p.blocks < 4) by *= p.blocks == 2 ? 0.93 : 0.96;
  if (cx.grouped)
    return by * (2.29 + 0.154 * sums + K * (0.259 * b + 0.218 * s + fill * (0.045 * b + 0.009 * s) +
                 whole * (0.160 * b + 0.139 * s) + more * 0.079 * sums) +
                 0.231 * more * sums + 0.52 * memory + 0.40 * beyond + wave * (0.062 * b + 0.134 * s) + 0.100 * simd * s);
  return by * (2.10 + 0.189 * sums + K * (0.309 * b + 0.177 * s + fill * (0.018 * b + 0.005 * s) +
                 whole * (0.203 * b + 0.085 * s) + more * 0.071 * sums) +
                 0.250 * more * sums + 0.71 * memory + 0.40 * beyond + (0.116 * wave + 0.067 * simd) * s);
}

// Fitted time (us) of the column-strip kernel with `cs` strips per workgroup.
// Up to 8 rows a launch costs 2.9 us.  A workgroup takes in its 8 cs k bytes
// of weights at about 28 GB/s, what its eight waves unpack and multiply, and
// workgroups beyond one per compute unit queue up behind each other, 0.4 us
// each; all together they draw 5.9 TB/s from memory at most.  Every workgroup
// also reads all rows of activations, which a compute unit takes from the L2s
// at about 73 GB/s.  Measured (M = 1, one strip): N = K = 2048 3.2 us, 4096 x
// 4096 4.3, N = 11008, K = 4096 7.8, N = 1024, K = 8192 5.5, N = 4096, K =
// 11008 7.5, 8192 x 8192 10.4 (two strips 9.1), N = 13824, K = 5120 11.4 (four
// strips 10.0); M = 16: 4096 x 4096 5.7, N = 11008, K = 4096 8.4, N = 4096, K = 11008 11.3.
// More rows are cut into parts of 16, a workgroup of the rows kernel per strip set and part.
double strip_cost(int m, int n, int k, int cs, const PlanCtx& cx) {
  const int cus = cx.cus;
  if (m > 16) return rows_cost(m, n, k, rows_pair(cs, 1), cx);
  const int wgs = ceil_div(n / 16, cs);
  if (m > 8) {
    // 9 to 16 rows, on the rows kernel: a launch, the strips' sums, what a workgroup takes in
    // and computes, dearer the fuller the chip, and workgroups beyond one per compute unit
    // (half way between the rounds they make and their share of one).  4981 launches over 1850
    // problems, 4 % rms
    const double K = k / 1000.0, r = (double)wgs / cus, fill = r < 1.0 ? r : 1.0;
    const double more = r > 1.0 ? 0.5 * (ceil_div(wgs, cus) + r) - 1.0 : 0.0;
    const double by = cs == 3 ? 1.055 : cs == 2 ? 1.0 : 1.03;
    if (cx.grouped)
      return by * (2.25 + 0.278 * cs + K * (0.168 + 0.119 * cs + 0.145 * fill * cs + more * (0.211 + 0.355 * cs)) +
                   0.32 * more + 0.0239 * m * K);
    return by * (2.23 + 0.252 * cs + K * (0.127 + 0.109 * cs + 0.130 * fill * cs + more * (0.257 + 0.327 * cs)) +
                 0.27 * more + 0.0266 * m * K);
  }
  // Up to 8 rows the constants are fitted on their own (M = 1, 4, 8: 7 % rms): the launch, the
  // rate a compute unit unpacks at, the rate it reads rows at, a queued
  // workgroup, and memory -- 5.85 TB/s while every round of workgroups fills
  // the compute units.
  const int per_cu = ceil_div(wgs, cus);
  const double last_round = wgs > cus ? (double)wgs / (per_cu * cus) : 1.0;
  const double by_cu = per_cu * 8.0 * cs * k / 28.0e3;
  const double by_memory = 0.5 * k * n / (5.85e6 * last_round);
  // (with fewer workgroups than compute units the rows come in sooner than this)
  const double rows = per_cu * 2.0 * m * k / 72.5e3 * (wgs < cus ? (0.5 + 0.5 * wgs / cus) : 1.0);
  // a wave's chunk is 256 / cs k-values (128 with three strips): a k range of
  // fewer than eight chunks leaves waves idle (K = 1024: one strip 0.2 to 0.3
  // us behind two at every N with 8 rows; fewer rows are no slower for it)
  const int chunks = ceil_div(k, cs == 3 ? 128 : 256 / cs);
  const double idle = m == 8 && chunks < 8 ? 0.7 * (1.0 - chunks / 8.0) : 0.0;
  // (a little of by_cu always: it decides between widths that memory bounds alike)
  return 2.88 + (by_cu > by_memory ? by_cu : by_memory) + rows + 0.43 * (per_cu - 1) + 0.02 * by_cu + idle;
}

// 16-column strips per workgroup of the column-strip kernel: the cheapest of
// 1, 2 and 4 where they divide n's strips, and for up to 16 rows of 3, which
// leaves the last workgroup with fewer (N = 11008, K = 4096, 230 workgroups
// of three strips against 172 of four: M = 8 8.2 against 8.5 us, M = 1 7.5 / 7.7
// with one strip; K = 8192: M = 1 12.3 against 13.6, M = 4 11.7 / 13.6; N = 5120,
// K = 5120: 10.3 against 8.4 with two)
// (0 where the planner's own rules leave none; a forced launch takes any)
int strips_per_workgroup(int m, int n, int k, const PlanCtx& cx) {
  const bool forced = cx.force.kernel == 3 || cx.force.strips != 0;
  int best = 0;
  double best_cost = 0.0;
  for (int cs = 1; cs <= 4; cs++) {
    // (three strips: not over k ranges of a chunk or two per wave, where their
    // three loads per chunk cost 8 % against two or four strips)
    if (cs == 3 ? ((m > 16 || k < 1024) && !forced) : n % (16 * cs) != 0) continue;
    // Rows in parts: at most two workgroups per compute unit (with three and
    // more the streaming kernel was 1.1 to 1.6 times faster wherever the fits,
    // its own 20 to 40 % high over short k ranges, promised otherwise: 48 rows
    // at N = 28672, K = 512 11.8 against 7.3 us, 64 rows at N = 11008, K = 2048
    // 13.5 against 11.2)
    if (m > 16 && !forced && ceil_div(n / 16, cs) * ceil_div(m, 16) > 2 * cx.cus) continue;
    if (cx.force.strips != 0 && cx.force.strips != cs && best != 0) continue;
    const double c = strip_cost(m, n, k, cs, cx);
    if (best == 0 || cx.force.strips == cs || c < best_cost) {
      best = cs;
      best_cost = c;
      if (cx.force.strips == cs) break;
    }
  }
  return best;
}

// The column-strip kernel against the other two: the streaming kernel reaches
// more of the memory's bandwidth (its workgroups share a column tile's k
// range, so every compute unit has work whatever n is), the strips pay nothing
// for the exchange between workgroups -- 2 us of a launch that takes 6.  The
// strips win while the weights are a few MiB per launch (M = 1: 4096 x 4096
// 4.3 against 6.3 us, N = 11008, K = 4096 8.5 against 9.7, N = 4096, K = 11008
// 7.5 against 9.1, 8192 x 8192 9.1 against 10.4, N = 28672, K = 8192 27.6
// against 23.9 -- there no more), 9 to 16 rows the same with a fit of its own for either kernel
// (over 3694 problems the choice takes 1.005 of the better of the two, 8 of them more than 10 %
// longer; by the fits of a kernel whose requests past the end made short ranges slow 1.018 and
// 210), and with more rows, in parts, while the parts fill the compute units at most twice (M =
// 100, N = 512, K = 1024 3.0 us; M = 41, N = 2304, K = 2048 4.6; M = 96, N = K = 4096 11.7 against
// 12.5 streaming, M = 1000, N = 256, K = 12416 17.8 against 22.7 on prefill tiles).
bool prefer_strips(int m, int n, int k, const PlanCtx& cx) {
  const int cs = strips_per_workgroup(m, n, k, cx);
  // (more rows over a deep k: what the rows kernel takes in the plan's place it takes for a pair
  // of its own, and the plan leaves strips by a margin)
  if (cs == 0) return false;
  const double strips = strip_cost(m, n, k, cs, cx) * (m > 16 && k >= 4096 ? 1.05 : 1.0);
  // Up to 8 rows with group scales over runs that straddle tiles the line lay here where it
  // cost least: over 74 such problems what it leaves takes 1.002 of the better of the two, by
  // equal costs 1.05 (4 x 21504 x 8192 22.8 us streaming, 19.5).  (Without group scales, and for
  // one strip per workgroup, one problem in three took 2 to 15 % longer by it.)
  const double line =
      m <= 8 && cx.grouped && cs > 1 && choose_stream_split(1, n, k, cx.cus).straddle ? 1.2 : 1.0;
  if (strips >= stream_cost_as_planned(m, n, k, cx) * line) return false;
  // (near prefill tiles the plan keeps those: the rows kernel, of which strips are a part, takes
  // their place where it is cheaper)
  return !(n % 256 == 0 && m > 48 && prefill_cost(m, n, k, cx) <= 1.03 * strips);
}

// Whether column strips may take the place of a streaming launch whose scratch cannot be had.
bool strips_instead(int m, int n, int k, const PlanCtx& cx) {
  if (m <= 8 || m > kStripMaxRows) return false;
  if (m <= 16) return true;
  const int cs = strips_per_workgroup(m, n, k, cx);
  return cs > 0 && strip_cost(m, n, k, cs, cx) <= 1.1 * stream_cost_as_planned(m, n, k, cx);
}

Plan make_plan(int m, int n, int k, int sms, const PlanCtx& cx) {
  Plan pl;
  // (the column-strip kernel does at most kStripMaxRows rows and takes no
  // hint: forced onto anything else it leaves the choice to the costs)
  const int force = cx.force.kernel == 3 && (m > kStripMaxRows || sms > 0) ? 0 : cx.force.kernel;
  // the prefill kernel's tiles are 256 columns wide (n is a multiple of 256
  // whenever m > 16, by the shape contract)
  const bool by_cost = force == 0 || force == 4;
  const bool prefill = n % 256 == 0 && (force == 2 || (by_cost && prefer_prefill(m, n, k, cx)));
  pl.ksplit = 1;
  pl.tile_rows = 0;
  pl.partial_bytes = 0;
  pl.row_parts = 1;
  pl.part_rows = 0;
  pl.strips = 0;
  if (m <= kStripMaxRows && sms <= 0 &&
      (force == 3 || (force == 0 && prefer_strips(m, n, k, cx)))) {
    pl.kernel = 3;
    pl.strips = strips_per_workgroup(m, n, k, cx);
    if (m > 16) {
      pl.row_parts = ceil_div(m, 16);
      pl.part_rows = 16;
    }
    pl.grid = ceil_div(n / 16, pl.strips) * pl.row_parts;
    pl.sp = make_stream_plan(n, k, 1);
    pl.launches = 1;
    return pl;
  }
  if (prefill) {
    // one workgroup per (tile of C, slice of k)
    pl.kernel = 2;
    pl.tile_rows = prefill_tile_rows(m, n, k, cx);
      const int tiles = ceil_div(m, pl.tile_rows) * (n / 256);
    pl.ksplit = prefill_k_slices(tiles, pl.tile_rows, k, cx);
    pl.grid = tiles * pl.ksplit;
    pl.sp = make_stream_plan(n, k, 1);
    pl.launches = 1;
    if (pl.ksplit > 1) pl.partial_bytes = (size_t)pl.grid * ceil_div(pl.tile_rows, 32) * 32 * 256 * 4;
    return pl;
  }
  pl.kernel = 1;
  const int rows = m < kStreamMaxRows ? m : kStreamMaxRows;
  const int mb = ceil_div(rows, 16);
  {
    // more than 64 rows: one launch with the rows cut into parts of 32 where
    // that is cheaper than a launch per 64 rows
    int parts = 0, wpt = 0, gpb = 0;
    const double cut = sms > 0 ? -1.0 : stream_parts_cost(m, n, k, cx, &parts, &wpt, &gpb);
    if (cut > 0.0 && (cx.force.row_halves == 2 || cut < stream_cost(m, n, k, cx.cus))) {
      pl.sp.NT = n / kTileN;
      pl.sp.KG = k / kGranuleK;
      pl.sp.gpb = gpb;
      pl.sp.wpt = wpt;
      pl.sp.grid = pl.sp.NT * parts * wpt;
      pl.row_parts = parts;
      pl.part_rows = 32;
      pl.grid = pl.sp.grid;
      pl.launches = 1;
      if (wpt > 1) pl.partial_bytes = (size_t)stream_slots(pl.sp) * stream_slot_bytes(2);
      return pl;
    }
  }
  if (sms > 0) {
    pl.sp = make_stream_plan(n, k, sms > kMaxStreamGrid ? kMaxStreamGrid : sms);
  } else {
    const StreamSplit split = choose_stream_split(mb, n, k, cx.cus);
    pl.sp.NT = n / kTileN;
    pl.sp.KG = k / kGranuleK;
    pl.sp.gpb = split.gpb;
    pl.sp.wpt = split.wpt;
    pl.sp.grid = split.wpt > 0 ? pl.sp.NT * split.wpt : ceil_div(pl.sp.NT * pl.sp.KG, split.gpb);
    // Many rows and many workgroups per tile: cut the rows in two instead of
    // the k range once more.  Each half is finished by half as many sharers,
    // with half the rows to sum, store and read back.
    const int half = 16 * ceil_div(ceil_div(rows, 2), 16);
    // the halves' own split: twice the tiles, half the row blocks
    const StreamSplit hs = choose_stream_split(half / 16, 2 * n, k, cx.cus);
    const bool can = m <= kStreamMaxRows && half < rows && split.wpt >= 2 && hs.wpt >= 1 &&
                     cx.counters >= 2;
    const bool want =
        can && (cx.force.row_halves == 2 ||
                (cx.force.row_halves == 0 &&
                 halves_gain(rows, 2 * hs.wpt, ceil_div(pl.sp.KG, 2 * hs.wpt)) > 0.25));
    if (want) {
      pl.row_parts = 2;
      pl.part_rows = half;
      pl.sp.wpt = hs.wpt;
      pl.sp.gpb = ceil_div(pl.sp.KG, pl.sp.wpt);
      pl.sp.grid = pl.sp.NT * 2 * pl.sp.wpt;
    }
  }
  pl.grid = pl.sp.grid;
  pl.launches = ceil_div(m, kStreamMaxRows);
  // column tiles that several workgroups share are finished through one
  // partial-sum slot per workgroup (cut tiles) or two (runs that may start and
  // end inside a tile)
  const bool shared = pl.sp.wpt > 0 ? pl.sp.wpt > 1 : pl.sp.gpb % pl.sp.KG != 0;
  if (shared)
    pl.partial_bytes = (size_t)stream_slots(pl.sp) *
                       stream_slot_bytes(pl.row_parts > 1 ? pl.part_rows / 16 : mb);
  return pl;
}

// The strips and row blocks of 16 of a workgroup of w4a16_rows.hip where that
// kernel computes the problem in place of the plan (strips 0: not).
struct RowsPlan {
  int strips, blocks;
};

// What the fit of streaming launches of 17 to 64 rows over k of 2048 and more is off by: it does
// not tell the kinds of scales apart, and knows little of how many workgroups share a tile (1108
// launches, by row blocks, cut in halves or not, and sharers: 2 to 4 % rms; 64 x 2048 x 8192,
// sixteen, 1.25 of the fit, 47 x 7168 x 9472, four, 0.93; tiles that are not shared by their depth:
// 17 x 28672 x 8192 1.03, a quarter of that 0.86).  And a line between these launches
// and the rows kernel costs least 2 % above, with three row blocks uncut at it.
double stream_off(int m, const Plan& pl, bool grouped) {
  const int sharers = pl.sp.wpt, blocks = ceil_div(m, 16);
  if (sharers == 0) return grouped ? 1.17 : 1.23;  // (runs that straddle tiles)
  double off;
  if (sharers == 1)
    off = pl.row_parts > 1 ? 0.94 : blocks == 2 ? 0.82 + 0.0017 * pl.sp.gpb : 0.80 + 0.001 * pl.sp.gpb;
  else if (pl.row_parts == 1)
    off = (blocks == 2 ? 1.02 : 0.925) + 0.006 * (sharers - 2);
  else if (sharers <= 8)
    off = 0.984 + 0.0133 * (sharers - 2);
  else  // (fetched in two rounds)
    off = blocks == 2 ? 1.07 : 1.173 + 0.0133 * (sharers - 9);
  return off * (grouped ? 1.0 : sharers > 8 ? 0.98 : pl.row_parts == 1 ? 0.955 : 0.935);
}

// For 17 rows and more, where it is cheaper than the plan.  Not over k ranges below 640, nor,
// with 16 rows per workgroup, below 2048, where the plan's column strips are that launch.  Over
// 6262 problems the choice takes 1.005 of the best launch measured, 37 of them more than 10 %
// longer (by a fit of a kernel whose weights went through registers, with factors: 1.016 and
// 355).  What the plans' own fits are off by near the line is in the limits; 0.03 to either side
// costs less than 0.001 of the time.
RowsPlan rows_plan(int m, int n, int k, int sms, const Plan& pl, const PlanCtx& cx) {
  if (cx.force.rows_strips > 0 && sms <= 0 && (cx.force.rows_strips < 8 || n % 128 == 0) &&
      rows_exist(cx.force.rows_strips, cx.force.rows_blocks, cx.grouped))
    return {cx.force.rows_strips, cx.force.rows_blocks};
  if (sms > 0 || m <= 16 || k < 640 || cx.force.any()) return {0, 0};
  double limit;
  if (pl.kernel == 1) {
    const double off = m > kStreamMaxRows ? (pl.sp.wpt == 1 ? 0.93 : cx.grouped ? 1.02 : 0.98)
                       : k < 2048         ? 1.03
                                          : stream_off(m, pl, cx.grouped);
    limit = stream_cost_as_planned(m, n, k, cx) * off;
  } else if (pl.kernel == 2) {
    // (rows far beyond an XCD's L2: 1316 x 512 x 5504 17.6 us, 18.3 on the rows kernel)
    limit = prefill_cost(m, n, k, cx) * (2e-6 * m * k > 8.0 ? 0.91 : 0.99);
  } else {
    limit = strip_cost(m, n, k, pl.strips, cx) * 1.0001;  // (up to three strips in parts are a pair of the list)
  }
  RowsPlan best = {0, 0};
  for (const RowsPair& p : kRowsPairs) {
    if (m <= 16 * (p.blocks - 1) || (p.blocks == 1 && k < 2048)) continue;  // (fewer blocks hold all rows)
    if (p.strips == 4 && (p.blocks == 1 || (p.blocks == 4 && !cx.grouped))) continue;  // (strips alone; does not exist)
    // (beyond what was fitted, and never the best there)
    if (ceil_div(n / 16, p.strips) * ceil_div(m, 16 * p.blocks) > 2.7 * cx.cus) continue;
    const double c = rows_cost(m, n, k, p, cx);
    if (c < limit) {
      best = {p.strips, p.blocks};
      limit = c;
    }
  }
  return best;
}

// A thread's last 32 plans, by everything that they are made from (no overrides among
// it): planning takes the host 0.6 to 2.6 us, most for 17 to 300 rows, and a decoder calls
// the same few sizes over and over.  The oldest makes room.  (One place for each size, by
// a hash, was found sooner but given to another size of the same place at every call of
// two such sizes: one set of four sizes in six.)
struct Planned {
  int m = 0, n = 0, k = 0, sms = 0, cus = 0, counters = 0;
  size_t partial_limit = 0;
  bool grouped = false;
  Plan plan;
  RowsPlan rows;
};
constexpr int kPlansKept = 32;
thread_local Planned t_plans[kPlansKept];
thread_local int t_oldest_plan = 0;

Planned make_plans(int m, int n, int k, int sms, const PlanCtx& cx) {
  Planned p;
  p.m = m;
  p.n = n;
  p.k = k;
  p.sms = sms;
  p.cus = cx.cus;
  p.counters = cx.counters;
  p.partial_limit = cx.partial_limit;
  p.grouped = cx.grouped;
  p.plan = make_plan(m, n, k, sms, cx);
  p.rows = rows_plan(m, n, k, sms, p.plan, cx);
  return p;
}

const Planned* kept_plans(int m, int n, int k, int sms, const PlanCtx& cx) {
  for (const Planned& p : t_plans)
    if (p.m == m && p.n == n && p.k == k && p.sms == sms && p.cus == cx.cus && p.counters == cx.counters &&
        p.partial_limit == cx.partial_limit && p.grouped == cx.grouped)
      return &p;
  return nullptr;
}

Planned plans_for(int m, int n, int k, int sms, const PlanCtx& cx) {
  if (cx.force.any()) return make_plans(m, n, k, sms, cx);
  const Planned* kept = kept_plans(m, n, k, sms, cx);
  if (kept) return *kept;
  Planned& place = t_plans[t_oldest_plan];
  t_oldest_plan = (t_oldest_plan + 1) % kPlansKept;
  return place = make_plans(m, n, k, sms, cx);
}

// Operands that 16-byte loads straight into LDS may fetch.  A tensor may start anywhere in its
// storage; loads to registers take any address, and that a load into LDS does is documented
// nowhere.
bool whole_lines(const void* A, const void* B) {
  return (((uintptr_t)A | (uintptr_t)B) & 15) == 0;
}

// The plan of a call whose operands do not start on 16 bytes, in place of one on the rows
// kernel: 9 to 16 rows stay column strips (enqueue launches them 8 at a time), more take
// 64-row prefill tiles, which load through registers, whole: nothing that a capture or a full
// pool could refuse.
Planned plans_off_lines(Planned p, PlanCtx cx) {
  const bool rows_kernel = p.rows.strips > 0 || (p.plan.kernel == 3 && p.m > 8);
  if (!rows_kernel) return p;
  p.rows = {0, 0};
  if (p.m > 16) {
    cx.partial_limit = 0;
    cx.force = Force();
    cx.force.kernel = 2;
    cx.force.tile_rows = 64;
    p.plan = make_plan(p.m, p.n, p.k, -1, cx);
  } else if (p.plan.kernel != 3) {
    cx.force = Force();
    cx.force.kernel = 3;
    p.plan = make_plan(p.m, p.n, p.k, -1, cx);
  }
  return p;
}

// Enqueue the launches of plan pl with the scratch of `view` (null pointers
// when the plan exchanges nothing through scratch).
int enqueue(const Plan& pl, const ScratchView& view, const void* A, const void* B, void* C,
            const void* s, int m, int n, int k, void* workspace, int groupsize, int max_par,
            hipStream_t stream) {
  // the caller's workspace holds at least n/128 * max_par zero ints
  // (reference marlin_gemm.cpp:29-31, marlin_cute_kernel.cu:68); one counter
  // per column tile is used (two where the rows are cut in halves: the plan
  // only does that when max_par >= 2), and the counters are spread max_par
  // ints apart (64 bytes at the launcher's default of 16)
  const int lock_stride = max_par > 16 ? 16 : max_par;
  (void)hipGetLastError();  // an earlier call's error is not this launch's
  int rc = MARLIN_OK;
  if (pl.kernel == 3) {
    // (off 16 bytes: up to 8 rows a launch, through registers)
    const int rows_per_launch = whole_lines(A, B) ? m : 8;
    for (int m0 = 0; m0 < m && rc == MARLIN_OK; m0 += rows_per_launch) {
      GemmArgs a = {};
      a.A = (const char*)A + (size_t)m0 * k * 2;
      a.B = B;
      a.C = (char*)C + (size_t)m0 * n * 2;
      a.S = s;
      a.M = m - m0 < rows_per_launch ? m - m0 : rows_per_launch;
      a.N = n;
      a.K = k;
      a.lock_stride = 1;
      a.row_parts = pl.row_parts;
      a.part_rows = pl.row_parts > 1 ? 16 : 0;
      rc = launch_strip(a, groupsize != -1, pl.strips, stream);
    }
  } else if (pl.kernel == 2) {
    GemmArgs a;
    a.A = A;
    a.B = B;
    a.C = C;
    a.S = s;
    a.M = m;
    a.N = n;
    a.K = k;
    a.locks = view.counters;
    a.lock_stride = kSliceCounterStride;
    a.scratch = view.partials;
    a.gpb = 0;
    a.wpt = 0;
    a.row_parts = 1;
    a.part_rows = 0;
    a.finish_polls = t_force.finish_polls < 0 ? kFinishPolls : t_force.finish_polls;
    // tiles of 80 to 128 rows: four waves with accumulators of all rows x 128 columns; 64-row tiles: eight
    // waves with 64 x 64
    rc = pl.tile_rows > 64 ? launch_prefill_wide(a, groupsize != -1, pl.tile_rows, pl.ksplit, stream)
                           : launch_prefill(a, groupsize != -1, pl.ksplit, stream);
  } else {
    // a launch per 64 rows, or one launch over all rows cut into parts
    const int rows_per_launch = pl.launches == 1 ? m : kStreamMaxRows;
    for (int m0 = 0; m0 < m && rc == MARLIN_OK; m0 += rows_per_launch) {
      GemmArgs a;
      a.A = (const char*)A + (size_t)m0 * k * 2;
      a.B = B;
      a.C = (char*)C + (size_t)m0 * n * 2;
      a.S = s;
      a.M = m - m0 < rows_per_launch ? m - m0 : rows_per_launch;
      a.N = n;
      a.K = k;
      a.locks = (int*)workspace;
      a.lock_stride = lock_stride;
      a.scratch = view.partials;
      a.gpb = pl.sp.gpb;
      a.wpt = pl.sp.wpt;
      a.row_parts = pl.row_parts;
      a.part_rows = pl.part_rows;
      rc = launch_stream(a, groupsize != -1, pl.grid, stream);
    }
  }
  if (rc == MARLIN_ERR_RUNTIME) set_error(w4a16::last_launch_error(), "kernel launch");
  return rc;
}

int enqueue_rows(const RowsPlan& rows, const void* A, const void* B, void* C, const void* s, int m,
                 int n, int k, int groupsize, hipStream_t stream) {
  (void)hipGetLastError();  // an earlier call's error is not this launch's
  GemmArgs a = {};
  a.A = A;
  a.B = B;
  a.C = C;
  a.S = s;
  a.M = m;
  a.N = n;
  a.K = k;
  const int rc = launch_rows(a, groupsize != -1, rows.strips, rows.blocks, stream);
  if (rc == MARLIN_ERR_RUNTIME) set_error(w4a16::last_launch_error(), "kernel launch");
  return rc;
}

// With `dev` current: this device's copy of the fixed scratch array.  Its
// counters need no clearing: the array is zero when the module is loaded and
// every launch hands its counters back zeroed.  (A clearing kernel on the first
// caller's stream could land in the middle of another stream's first launch.)
unsigned char* static_scratch_for(int dev) {
  std::lock_guard<std::mutex> lk(g_mu);
  DeviceState& d = g_dev[dev];
  if (d.static_scratch) return d.static_scratch;
  void* ptr = nullptr;
  hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) {
    set_error(e, "hipGetSymbolAddress(scratch)");
    return nullptr;
  }
  d.static_scratch = (unsigned char*)ptr;
  return d.static_scratch;
}

// use_static: marlin_gemm_static -- the fixed array instead of the pool, a
// plan made for its size, and no allocation on any path.
int run(const void* A, const void* B, void* C, const void* s, int m, int n, int k,
        void* workspace, int groupsize, int dev, hipStream_t stream, int thread_k, int thread_n,
        int sms, int max_par, bool use_static) {
  int rc = check_shape(m, n, k, groupsize, thread_k, thread_n);
  if (rc != MARLIN_OK || m == 0 || n == 0 || k == 0) return rc;
  if (max_par < 1) {
    // the tile counters live in the caller's workspace, max_par ints apart
    snprintf(g_last_error, sizeof(g_last_error), "max_par = %d: must be at least 1", max_par);
    return MARLIN_ERR_WORKSPACE;
  }
  // the kernels address A, B and C with 32-bit byte offsets
  const long long lim = 0x7fffffffLL;
  if ((long long)k * n / 2 > lim || (long long)m * k * 2 > lim || (long long)m * n * 2 > lim) {
    snprintf(g_last_error, sizeof(g_last_error),
             "operand of more than 2 GiB (m=%d n=%d k=%d): split the call", m, n, k);
    return MARLIN_ERR_RUNTIME;
  }
  if (dev < 0 || dev >= kMaxDevices) {
    snprintf(g_last_error, sizeof(g_last_error), "device index %d out of range", dev);
    return MARLIN_ERR_RUNTIME;
  }
  int prev = -1;
  hipError_t e = hipGetDevice(&prev);
  if (e != hipSuccess) {
    set_error(e, "hipGetDevice");
    return MARLIN_ERR_RUNTIME;
  }
  if (prev != dev && (e = hipSetDevice(dev)) != hipSuccess) {
    set_error(e, "hipSetDevice");
    return MARLIN_ERR_RUNTIME;
  }
  const int cus = device_cus(dev);
  rc = MARLIN_ERR_RUNTIME;
  if (cus > 0 && configure_device(dev)) {
    PlanCtx cx = {cus, use_static ? kStaticPartialBytes : kPoolPartialLimit, t_force, groupsize != -1};
    cx.counters = max_par > 16 ? 16 : max_par;  // the counters of a tile sit that many ints apart
    Planned planned = plans_for(m, n, k, sms, cx);
    if (!whole_lines(A, B)) planned = plans_off_lines(planned, cx);
    Plan pl = planned.plan;
    ScratchView view = {nullptr, nullptr};
    bool ok = true;
    if (use_static) {
      if (pl.partial_bytes > kStaticPartialBytes) {
        snprintf(g_last_error, sizeof(g_last_error),
                 "marlin_gemm_static: this call (m=%d n=%d k=%d sms=%d) needs %zu bytes of "
                 "partial sums, the fixed scratch holds %zu: use marlin_gemm",
                 m, n, k, sms, pl.partial_bytes, kStaticPartialBytes);
        ok = false;
      } else if (pl.partial_bytes > 0) {
        unsigned char* base = static_scratch_for(dev);
        ok = base != nullptr;
        if (ok) {
          view.counters = (int*)base;
          view.partials = (float*)(base + kCounterBytes);
        }
      }
    } else if (pl.partial_bytes > 0) {
      ok = scratch_acquire(dev, stream, pl.partial_bytes, &view, g_last_error,
                           sizeof(g_last_error));
      if (!ok && pl.kernel == 2) {
        // slices of prefill tiles are there for speed alone: where their scratch
        // cannot be had (a stream under capture, a full pool) the problem is
        // computed without any
        cx.partial_limit = 0;
        pl = make_plan(m, n, k, sms, cx);
        if (pl.partial_bytes > 0) {
          cx.force.kernel = 2;
          pl = make_plan(m, n, k, sms, cx);
        }
        ok = pl.partial_bytes == 0;
      } else if (!ok && pl.kernel == 1 && sms <= 0 && !cx.force.any() && strips_instead(m, n, k, cx)) {
        // and streaming launches of 9 to 16 rows, or of more where the line between the two is
        // a matter of a tenth, by column strips: where it lies moves with either kernel's speed
        cx.force.kernel = 3;
        pl = make_plan(m, n, k, sms, cx);
        ok = pl.partial_bytes == 0;
      }
    }
    // (with the plan's scratch in hand: what a stream must have seen before it can be
    // captured does not depend on a choice that is a matter of speed)
    if (ok && planned.rows.strips > 0)
      rc = enqueue_rows(planned.rows, A, B, C, s, m, n, k, groupsize, stream);
    else if (ok)
      rc = enqueue(pl, view, A, B, C, s, m, n, k, workspace, groupsize, max_par, stream);
  }
  if (prev != dev) (void)hipSetDevice(prev);
  return rc;
}

}  // namespace

extern "C" {

int marlin_gemm(const void* A, const void* B, void* C, const void* s, int prob_m, int prob_n,
                int prob_k, void* workspace, int groupsize, int dev, void* stream, int thread_k,
                int thread_n, int sms, int max_par) {
  return run(A, B, C, s, prob_m, prob_n, prob_k, workspace, groupsize, dev, (hipStream_t)stream,
             thread_k, thread_n, sms, max_par, false);
}

int marlin_cute(const void* A, const void* B, void* C, void* s, int prob_m, int prob_n,
                int prob_k, void* workspace, int groupsize, int dev, void* stream, int thread_k,
                int thread_n, int sms, int max_par) {
  return marlin_gemm(A, B, C, s, prob_m, prob_n, prob_k, workspace, groupsize, dev, stream,
                     thread_k, thread_n, sms, max_par);
}

int marlin_official(const void* A, const void* B, void* C, void* s, int prob_m, int prob_n,
                    int prob_k, void* workspace, int groupsize, int dev, void* stream,
                    int thread_k, int thread_n, int sms, int max_par) {
  return marlin_gemm(A, B, C, s, prob_m, prob_n, prob_k, workspace, groupsize, dev, stream,
                     thread_k, thread_n, sms, max_par);
}

int marlin_gemm_static(const void* A, const void* B, void* C, const void* s, int prob_m,
                       int prob_n, int prob_k, void* workspace, int groupsize, int dev,
                       void* stream, int thread_k, int thread_n, int sms, int max_par) {
  return run(A, B, C, s, prob_m, prob_n, prob_k, workspace, groupsize, dev, (hipStream_t)stream,
             thread_k, thread_n, sms, max_par, true);
}

long long marlin_gemm_static_capacity(void) { return (long long)kStaticPartialBytes; }

int marlin_mul(const void* A, const void* B, void* C, const void* s, int prob_m, int prob_n,
               int prob_k, int s_rows, void* workspace, long long workspace_numel, int dev,
               void* stream, int thread_k, int thread_n, int sms, int max_par, int cute_version,
               char* err, int err_len) {
  (void)cute_version;  // one implementation serves both reference variants
  auto fail = [&](int code, const char* fmt, auto... args) {
    if (err && err_len > 0) snprintf(err, (size_t)err_len, fmt, args...);
    return code;
  };
  if (err && err_len > 0) err[0] = 0;
  if (s_rows <= 0) return fail(MARLIN_ERR_GROUPS, "k=%d not compatible with %d groups.", prob_k, s_rows);
  int groupsize = s_rows == 1 ? -1 : prob_k / s_rows;
  if (groupsize != -1 && groupsize * s_rows != prob_k)
    return fail(MARLIN_ERR_GROUPS, "k=%d not compatible with %d groups.", prob_k, s_rows);
  // (the reference's comparison, marlin_gemm.cpp:29-31, lets any workspace pass
  // when max_par < 1; the tile counters need at least one int per tile)
  const int par = max_par < 1 ? 1 : max_par;
  if (workspace_numel < (long long)(prob_n / 128) * par)
    return fail(MARLIN_ERR_WORKSPACE, "workspace must be of size at least %d.",
                prob_n / 128 * par);
  int rc = marlin_gemm(A, B, C, s, prob_m, prob_n, prob_k, workspace, groupsize, dev, stream,
                       thread_k, thread_n, sms, par);
  if (rc == MARLIN_ERR_PROB_SHAPE)
    return fail(rc, "Problem (m=%d, n=%d, k=%d) not compatible with thread_k=%d, thread_n=%d.",
                prob_m, prob_n, prob_k, thread_k, thread_n);
  if (rc == MARLIN_ERR_KERN_SHAPE)
    return fail(rc, "No kernel implementation for thread_k=%d, thread_n=%d, groupsize=%d.",
                thread_k, thread_n, groupsize);
  if (rc == MARLIN_ERR_RUNTIME) return fail(rc, "HIP runtime error: %s", g_last_error);
  if (rc != MARLIN_OK) return fail(rc, "%s", g_last_error);
  return rc;
}

int marlin_amd_check(int prob_m, int prob_n, int prob_k, int groupsize, int thread_k,
                     int thread_n) {
  return check_shape(prob_m, prob_n, prob_k, groupsize, thread_k, thread_n);
}

int marlin_amd_plan(int prob_m, int prob_n, int prob_k, int groupsize, int thread_k,
                    int thread_n, int sms, int cus, int* out) {
  for (int i = 0; i < 13; i++) out[i] = 0;
  int rc = check_shape(prob_m, prob_n, prob_k, groupsize, thread_k, thread_n);
  if (rc != MARLIN_OK || prob_m == 0 || prob_n == 0 || prob_k == 0) return rc;
  const PlanCtx cx = {cus, kPoolPartialLimit, t_force, groupsize != -1};
  Plan pl = make_plan(prob_m, prob_n, prob_k, sms, cx);
  out[0] = pl.kernel;
  out[1] = pl.grid;
  out[2] = pl.sp.gpb;
  out[3] = pl.sp.NT;
  out[4] = pl.sp.KG;
  out[5] = pl.launches;
  out[6] = pl.ksplit;
  out[7] = pl.tile_rows;
  out[8] = pl.kernel == 1 ? pl.sp.wpt : 0;
  out[9] = (int)(pl.partial_bytes >> 10);
  out[10] = pl.kernel == 1 || pl.kernel == 3 ? pl.row_parts : 1;
  out[11] = pl.kernel == 1 || pl.kernel == 3 ? pl.part_rows : 0;
  out[12] = pl.strips;
  return rc;
}

int marlin_amd_rows_plan(int prob_m, int prob_n, int prob_k, int groupsize, int cus, int* out) {
  out[0] = out[1] = 0;
  int thread_k = -1, thread_n = -1;
  int rc = check_shape(prob_m, prob_n, prob_k, groupsize, thread_k, thread_n);
  if (rc != MARLIN_OK || prob_m == 0 || prob_n == 0 || prob_k == 0) return rc;
  const PlanCtx cx = {cus, kPoolPartialLimit, t_force, groupsize != -1};
  const RowsPlan rows =
      rows_plan(prob_m, prob_n, prob_k, -1, make_plan(prob_m, prob_n, prob_k, -1, cx), cx);
  out[0] = rows.strips;
  out[1] = 16 * rows.blocks;
  return rc;
}

int marlin_amd_plan_kept(int prob_m, int prob_n, int prob_k, int groupsize, int cus) {
  int thread_k = -1, thread_n = -1;
  const int rc = check_shape(prob_m, prob_n, prob_k, groupsize, thread_k, thread_n);
  if (rc != MARLIN_OK || prob_m == 0 || prob_n == 0 || prob_k == 0) return -1;
  const PlanCtx cx = {cus, kPoolPartialLimit, t_force, groupsize != -1};
  if (kept_plans(prob_m, prob_n, prob_k, -1, cx)) return 1;
  plans_for(prob_m, prob_n, prob_k, -1, cx);
  return 0;
}

int marlin_amd_plan_costs(int prob_m, int prob_n, int prob_k, int groupsize, int cus, double* out) {
  for (int i = 0; i < 4; i++) out[i] = -1.0;
  int thread_k = -1, thread_n = -1;
  int rc = check_shape(prob_m, prob_n, prob_k, groupsize, thread_k, thread_n);
  if (rc != MARLIN_OK || prob_m == 0 || prob_n == 0 || prob_k == 0) return rc;
  const PlanCtx cx = {cus, kPoolPartialLimit, t_force, groupsize != -1};
  out[0] = stream_cost_as_planned(prob_m, prob_n, prob_k, cx);
  if (prob_n % 256 == 0) out[1] = prefill_cost(prob_m, prob_n, prob_k, cx);
  if (prob_m <= kStripMaxRows) {
    const int cs = strips_per_workgroup(prob_m, prob_n, prob_k, cx);
    if (cs > 0) out[2] = strip_cost(prob_m, prob_n, prob_k, cs, cx);
    out[3] = cs;
  }
  return rc;
}

void marlin_amd_force_kernel(int which) { t_force.kernel = which >= 1 && which <= 4 ? which : 0; }
void marlin_amd_force_strips(int strips) {
  t_force.strips = strips >= 1 && strips <= 4 ? strips : 0;
}

void marlin_amd_force_k_slices(int slices) { t_force.k_slices = slices > 0 ? slices : 0; }

void marlin_amd_force_row_halves(int mode) { t_force.row_halves = mode == 1 || mode == 2 ? mode : 0; }

void marlin_amd_force_tile_rows(int rows) {
  t_force.tile_rows = rows >= 64 && rows <= 128 && rows % 16 == 0 ? rows : 0;
}

void marlin_amd_force_rows(int strips, int blocks) {
  const bool exists = rows_exist(strips, blocks, true);  // (a pair of one scale per column has one of groups)
  t_force.rows_strips = strips < 0 ? -1 : exists ? strips : 0;
  t_force.rows_blocks = exists ? blocks : 0;
}

void marlin_amd_force_finish_polls(int polls) {
  t_force.finish_polls = polls < 0 || polls > kFinishPolls ? -1 : polls;
}

void marlin_amd_work_order(int grid, int* out) {
  for (int b = 0; b < grid; b++) out[b] = xcd_work_index(b, grid);
}

long long marlin_amd_scratch_bytes(int dev, int* buffers) {
  return (long long)scratch_bytes_held(dev, buffers);
}

long long marlin_amd_release(int dev) { return (long long)scratch_release(dev); }

int marlin_amd_device_info(int dev, int* out) {
  const hipDeviceAttribute_t what[5] = {
      hipDeviceAttributeMultiprocessorCount, hipDeviceAttributeClockRate,
      hipDeviceAttributeMemoryClockRate, hipDeviceAttributeMemoryBusWidth,
      hipDeviceAttributeL2CacheSize};
  for (int i = 0; i < 5; i++) {
    out[i] = 0;
    hipError_t e = hipDeviceGetAttribute(&out[i], what[i], dev);
    if (e != hipSuccess) {
      set_error(e, "hipDeviceGetAttribute");
      return MARLIN_ERR_RUNTIME;
    }
  }
  return MARLIN_OK;
}

const char* marlin_amd_last_error(void) { return g_last_error; }

const char* marlin_amd_version(void) { return "marlin_amd 0.2 (gfx950)"; }

}  // extern "C"
