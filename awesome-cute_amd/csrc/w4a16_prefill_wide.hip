// Prefill W4A16 kernel with one wave per SIMD: 128-row x 256-column tiles of C
// for launches that are bound by the matrix pipe and by what competes with it,
// and tiles of 112, 96 and 80 rows for row counts that would leave much of a
// 64- or 128-row tile empty.  A step of the main loop takes a 112-row tile 0.93,
// a 96-row tile 0.86 and an 80-row tile 0.80 of a 128-row tile's time: what is
// spared is matrix time and power, the unpack stays (M = 300, N = 28672, K =
// 8192: 300 rows as 3 x 128 172 us, as 4 x 80 142).
//
// A workgroup of four waves owns a 128 x 256 tile (and, like the other prefill
// kernel, one of `ksplit` slices of the k range when tiles alone would leave
// compute units idle).  Wave (nw, kh) computes the 128-column half nw of the
// tile over the k half kh of the workgroup's range: a 128 x 128 fp32
// accumulator, all 256 AGPRs, which is why there is one wave per SIMD.  The
// two k halves are added through LDS at the end.
//
// With k slices the rest is latency: at M = 128, N = K = 4096 in eight slices
// the loop ends at 9 us, the k halves take 0.5, the partial sums out 2.3, the
// other slices' arrival 1.8 and adding up and writing the tile 4.  Finished by
// the last arrival alone the launch took 26.3 us, by all slices together 18.0
// (four slices 23.5 / 20.0; two, M = 1024, 37.8 / 35.8).
//
// What this shape buys over eight waves with 128 x 64 accumulators:
//   - The packed weights never pass through LDS.  A wave's 128 columns are two
//     whole 64-column Marlin blocks, so MFMA lane (kg, nu) loads the 16-byte
//     piece of Marlin lane (t = kg, c = nu%8) of block nu/8 straight into
//     registers (coalesced: a wave instruction reads 1 KiB of one packed row),
//     and its four words are the operands of the four 16-column groups.
//   - Every activation operand read from LDS (one ds_read_b128) feeds eight
//     MFMAs instead of four, and every unpacked weight word still meets all
//     eight row blocks.
// Per 32-deep k step a wave issues 64 MFMAs, 8 LDS operand reads, 2 weight
// loads and the unpack of 8 packed words (104 VALU instructions with group
// scales), dealt out two behind every MFMA; the activation slab of a 64-deep
// stage (128 rows, staged through registers into two LDS slabs per k half, in
// the k-slot order of the weight layout) costs a thread 8 loads and 16 LDS
// writes per 128 MFMAs.
//
// Prologue, main loop and the hand-over of the accumulators are one assembly
// statement with fixed registers, written by gen_prefill_wide.py (which also
// documents the register map and the schedule); the build runs it.  The code
// here computes what the statement takes in and finishes the tile.
#include <type_traits>

#include "buffer_loads.hpp"
#include "w4a16_common.hpp"

namespace w4a16 {

namespace {

constexpr int kWdTileN = 256;
constexpr int kWdRing = 2;                    // activation slabs in LDS per k half
constexpr int kWdPitch = kWdTileN * 2 + 16;   // fp16 tile row in LDS on the way out

// what follows from the row blocks of 16 of a tile (RB = 5 to 8)
template <int RB>
struct WdShape {
  static constexpr int kTileM = 16 * RB;
  static constexpr int kHB = (RB + 1) / 2;  // row blocks a k half finishes (the second one RB - kHB)
  static constexpr int kPlane = kTileM * 16;               // one k group of a step: rows x 16 bytes
  static constexpr int kStepBytes = 4 * kPlane + 128;      // one 32-deep k step of a slab (+pad)
  static constexpr int kSlabBytes = 2 * kStepBytes;        // a 64-deep stage
  static constexpr int kRingBytes = kWdRing * kSlabBytes;  // per k half
  // the epilogue reuses the rings: 4 waves x kHB row blocks x 8 KiB of fp32 to
  // swap between the k halves, then the fp16 tile with padded rows
  static constexpr int kSwapBytes = 4 * kHB * 8 * 1024;
  static constexpr int kLdsBytes = kSwapBytes > 2 * kRingBytes ? kSwapBytes : 2 * kRingBytes;
  static_assert(kTileM * kWdPitch <= kLdsBytes, "");
  static constexpr int kPartBytes = kSwapBytes;  // fp32 sums of a tile in scratch
};

}  // namespace

// SLICED: with k slices of other workgroups.  Kernels of their own for whole
// tiles: in one kernel for both, the sums of a whole tile took moves and tests
// on the way out (M = 3614, N = 6656, K = 1280 with one scale per column 58.0
// -> 59.3 us).
template <bool GROUP, int RB, bool SLICED>
__global__ __launch_bounds__(256) void prefill_wide_kernel(GemmArgs p, int tiles_m, int tiles_n,
                                                           int ksplit) {
  extern __shared__ __attribute__((aligned(16))) char smem_all[];  // Shape::kLdsBytes
  __shared__ int s_shares;
  {
    // fetch every kernel argument in one round trip
    const void *a_ = p.A, *b_ = p.B, *s_ = p.S;
    void* c_ = p.C;
    int* l_ = p.locks;
    float* sc_ = p.scratch;
    asm volatile("" ::"s"(a_), "s"(b_), "s"(s_), "s"(c_), "s"(l_), "s"(sc_), "s"(p.M), "s"(p.N),
                 "s"(p.K), "s"(tiles_m), "s"(tiles_n), "s"(ksplit));
  }
  using Shape = WdShape<RB>;
  constexpr int HB = Shape::kHB;
  constexpr int kWdTileM = Shape::kTileM;

  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int kh = wave >> 1;  // k half
  const int nw = wave & 1;   // 128-column half of the tile
  const int tid = threadIdx.x & 127;  // thread within the k half
  const int lane = threadIdx.x & 63;
  const int kg = lane >> 4;
  const int nu = lane & 15;
  char* smem = smem_all + kh * Shape::kRingBytes;

  // Same numbering of the work as the other prefill kernel: every XCD
  // (workgroup id mod 8) gets a contiguous run of tile numbers, tiles are
  // numbered in panels of 8 column tiles with the row tile next, and the k slices
  // of a tile are consecutive work indices: they meet behind one L2.  (With slices
  // dealt out one by one where their number is no multiple of 8, over M = 33 ...
  // 8192, K < 6144: 1.09 times the time.)  Whole tiles of eight columns or more
  // get runs only if their number is a multiple of 8 (else no difference on
  // average, up to 6 % either way); of fewer, always, so that the columns of a row
  // tile read A from one L2 (N = 256 ... 1792, M = 600 ... 8192: 1.02 times the time
  // without, 1.05 with more tiles than compute units).
  const int total = tiles_m * tiles_n * ksplit;
  const bool runs = SLICED || (total & 7) == 0 || tiles_n < 8;
  const int work = runs ? xcd_work_index((int)blockIdx.x, total) : (int)blockIdx.x;
  const int tile = SLICED ? work / ksplit : work;
  const int ks = SLICED ? work - tile * ksplit : 0;
  int tm, tn;
  if ((tiles_n & 7) == 0) {
    const int per_panel = 8 * tiles_m;
    const int panel = tile / per_panel, within = tile - panel * per_panel;
    tm = within >> 3;
    tn = panel * 8 + (within & 7);
  } else {
    tm = tile / tiles_n;
    tn = tile - tm * tiles_n;
  }
  const int m0 = tm * kWdTileM;
  const int rows = min(kWdTileM, p.M - m0);

  // raw buffer resources (base, no stride, bytes, flags) as the words the
  // assembly takes; the A resource covers the rows of this tile only
  const i4 rb_words = rsrc_words(p.B, (unsigned)p.K * (unsigned)(p.N / 2));
  const i4 rs_words = rsrc_words(p.S, (unsigned)(GROUP ? p.K / 128 : 1) * (unsigned)p.N * 2u);
  i4 ra_words =
      rsrc_words((const char*)p.A + (size_t)m0 * p.K * 2, (unsigned)rows * (unsigned)p.K * 2u);
  const int b_row = p.N * 8;  // bytes per packed row (16 k of every column)

  // packed weights: piece of Marlin lane (t = kg, c = nu%8) of block 2nw + nu/8
  const int b_lane = 2048 * tn + 1024 * nw + 64 * nu + 16 * kg;
  // group scales: the 8 halfs at 8*nu of the permuted row are those of columns
  // 64(nu/8) + 16j + 8h + nu%8, in the order 2j + h
  const int s_lane = (256 * tn + 128 * nw) * 2 + 16 * nu;

  // slab staging: thread (row = tid/8 + 16 i', chunk x = tid%8) moves 16 bytes,
  // i' = (i + HB kh) % RB: the second k half keeps its row blocks rotated by HB,
  // so that in both halves the first accumulator blocks are the ones the wave
  // finishes (HB of them; RB - HB in the second half) and the last HB hold the
  // ones it hands to the other half.  Rows past the end of A read as zeros
  // (out-of-range buffer offset).
  const int ax = tid & 7;
  int a_lane[RB];
#pragma unroll
  for (int i = 0; i < RB; i++) {
    const int at = i + HB * kh;
    const int r = (tid >> 3) + 16 * (at >= RB ? at - RB : at);
    a_lane[i] = r < rows ? r * p.K * 2 + 16 * ax : kOob;
  }
  // LDS slab: [step][k group][row][slot] dwords; chunk x -> step x/4, slot x%4
  const int lds_wr =
      (int)(size_t)(smem + (ax >> 2) * Shape::kStepBytes + (tid >> 3) * 16 + (ax & 3) * 4);
  const int lds_rd = (int)(size_t)(smem + kg * Shape::kPlane + nu * 16);
  // where this wave leaves its last accumulator blocks for the other k half
  const int lds_swap = (int)(size_t)(smem_all + wave * (HB * 8 * 1024) + lane * 16);

  // this half's stages: [s_begin, s_end) of the K/64 stages; the loop runs the
  // same count in both halves (a stage past s_end fetches zeros)
  const int stages_all = p.K / 64;
  const int st0 = (int)((unsigned)ks * (unsigned)stages_all / (unsigned)ksplit);
  const int st1 = (int)((unsigned)(ks + 1) * (unsigned)stages_all / (unsigned)ksplit);
  const int half_stages = (st1 - st0 + 1) >> 1;
  const int s_begin = st0 + kh * half_stages;
  const int s_end = kh ? st1 : st0 + half_stages;
  const int stages = half_stages;
  const int s_row = p.N * 2;  // bytes per row of group scales

  f4 fin[HB][8];  // the first accumulator blocks: row blocks own, own+1, ... of the tile
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (GROUP && RB == 8) {
#include "w4a16_prefill_wide_group128.inc"
  } else if constexpr (GROUP && RB == 7) {
#include "w4a16_prefill_wide_group112.inc"
  } else if constexpr (GROUP && RB == 6) {
#include "w4a16_prefill_wide_group96.inc"
  } else if constexpr (GROUP) {
#include "w4a16_prefill_wide_group80.inc"
  } else if constexpr (RB == 8) {
#include "w4a16_prefill_wide_chan128.inc"
  } else if constexpr (RB == 7) {
#include "w4a16_prefill_wide_chan112.inc"
  } else if constexpr (RB == 6) {
#include "w4a16_prefill_wide_chan96.inc"
  } else {
#include "w4a16_prefill_wide_chan80.inc"
  }
#else  // the host pass only needs the launch stub
  (void)rb_words, (void)rs_words, (void)ra_words, (void)b_row, (void)b_lane, (void)s_lane;
  (void)lds_wr, (void)lds_rd, (void)lds_swap, (void)s_begin, (void)s_end, (void)stages;
  (void)s_row, (void)a_lane;
  for (auto& r : fin)
    for (auto& v : r) v = (f4){0.f, 0.f, 0.f, 0.f};
#endif
  // the other k half's sums of the same row blocks
  __syncthreads();
  const int own = HB * kh;  // first row block this wave finishes
  {
    // (with an odd number of row blocks the second half's are one slot further
    // on, and it finishes one fewer)
    const f4* in = (const f4*)smem_all + (size_t)(wave ^ 2) * (HB * 8 * 64) +
                   (kh ? (2 * HB - RB) * 8 * 64 : 0);
#pragma unroll
    for (int i = 0; i < HB; i++) {
      if ((RB & 1) && own + i >= RB) continue;
#pragma unroll
      for (int o = 0; o < 8; o++) fin[i][o] += in[(i * 8 + o) * 64 + lane];
    }
  }

  // ---- k slices of other workgroups: every slice writes the fp32 sums that
  // others will add up through to memory (whole 1 KiB lines per wave
  // instruction), waits for the acknowledgement and arrives; the slices then
  // finish the tile together.  Piece e of it is half the columns (operands
  // 4 (e%2) ... +3) of row block e/2 of every wave; all slices of it are added
  // in slice order, this one's from registers at its place in that order.
  constexpr int NP = 2 * HB;
  int pieces = (1 << NP) - 1;
  if constexpr (SLICED) {
    constexpr int part_bytes = Shape::kPartBytes;
    const __amdgpu_buffer_rsrc_t rP = make_rsrc(p.scratch, 0x7fffffffu);
    int* const word = &p.locks[tile * p.lock_stride];
    const int at = (wave * (HB * 8) * 64 + lane) * 16;
    auto write_out = [&](int which) {
#pragma unroll
      for (int e = 0; e < NP; e++) {
        if (!(which >> e & 1)) continue;
#pragma unroll
        for (int o = 4 * (e & 1); o < 4 * (e & 1) + 4; o++)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, fin[e >> 1][o]), rP,
                                                 at + ((e >> 1) * 8 + o) * 1024, work * part_bytes,
                                                 16 /* sc1 */);
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): my stores have been acknowledged
      __syncthreads();
    };
    const int my_share = finish_pieces(1 << ks, ksplit, NP);
    write_out(pieces & ~my_share);
    if (threadIdx.x == 0) s_shares = finish_arrive(word, ksplit, ks, p.finish_polls);
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_shares) == 0) {
      write_out(my_share);
      if (threadIdx.x == 0) s_shares = finish_abandon(word, ksplit, ks);
      __syncthreads();
    }
    pieces = __builtin_amdgcn_readfirstlane(finish_pieces(s_shares, ksplit, NP));
    // what is requested at once: a row block of up to four slices, else half of one
    auto add_up = [&](auto SL, auto NO, int i, int o0) {
      constexpr int sl = decltype(SL)::value, no = decltype(NO)::value;
      f4 v[sl][no];
#pragma unroll
      for (int k2 = 0; k2 < sl; k2++) {
        if (k2 >= ksplit || k2 == ks) continue;
#pragma unroll
        for (int o = 0; o < no; o++)
          v[k2][o] = __builtin_bit_cast(
              f4, __builtin_amdgcn_raw_buffer_load_b128(rP, at + (i * 8 + o0 + o) * 1024,
                                                        (tile * ksplit + k2) * part_bytes, 16 /* sc1 */));
      }
#pragma unroll
      for (int o = 0; o < no; o++) {
        f4 sum = ks == 0 ? fin[i][o0 + o] : v[0][o];
#pragma unroll
        for (int k2 = 1; k2 < sl; k2++)
          if (k2 < ksplit) sum += k2 == ks ? fin[i][o0 + o] : v[k2][o];
        fin[i][o0 + o] = sum;
      }
    };
    using std::integral_constant;
#pragma unroll
    for (int i = 0; i < HB; i++) {
      const int both = pieces >> (2 * i) & 3;
      if (both == 3 && ksplit <= 4) {
        add_up(integral_constant<int, 4>{}, integral_constant<int, 8>{}, i, 0);
      } else {
        if (both & 1) add_up(integral_constant<int, 8>{}, integral_constant<int, 4>{}, i, 0);
        if (both & 2) add_up(integral_constant<int, 8>{}, integral_constant<int, 4>{}, i, 4);
      }
    }
  }
  __syncthreads();

  // fp16 tile -> LDS in row-major order, then whole 512-byte rows go out with
  // coalesced 16-byte stores.  A lane holds row 16 i + nu and, per operand
  // (j, h), the four consecutive columns 64(q/2) + 16j + 8h + 4(q%2) + r of its
  // wave's 128, q = lane/16.
  const int q = lane >> 4;
#pragma unroll
  for (int o = 0; o < 8; o++) {
    const int nloc = 128 * nw + 64 * (q >> 1) + 16 * (o >> 1) + 8 * (o & 1) + 4 * (q & 1);
    h4 sc = {(half_t)1.f, (half_t)1.f, (half_t)1.f, (half_t)1.f};
    if (!GROUP) {
      const half_t* S = (const half_t*)p.S;
#pragma unroll
      for (int r = 0; r < 4; r++) sc[r] = S[scale_index_single(kWdTileN * tn + nloc + r)];
    }
#pragma unroll
    for (int i = 0; i < HB; i++) {
      if ((RB & 1) && own + i >= RB) continue;
      if (SLICED && !(pieces >> (2 * i + (o >> 2)) & 1)) continue;
      const int m = 16 * (own + i) + nu;
      h4 v = {(half_t)fin[i][o][0], (half_t)fin[i][o][1], (half_t)fin[i][o][2],
              (half_t)fin[i][o][3]};
      if (!GROUP) v *= sc;
      *(h4*)(smem_all + m * kWdPitch + nloc * 2) = v;
    }
  }
  __syncthreads();
  half_t* C = (half_t*)p.C;
#pragma unroll
  for (int it = 0; it < kWdTileM / 8; it++) {
    const int piece = it * 256 + (int)threadIdx.x;  // 16-byte piece of the tile
    const int m = piece >> 5;
    const int c16 = piece & 31;
    // (row block i of either k half; columns 32 ... 63 of every 64: operands 4 to 7)
    const int i = m >= 16 * HB ? (m >> 4) - HB : m >> 4;
    if (m < rows && (!SLICED || (pieces >> (2 * i + ((c16 >> 2) & 1)) & 1))) {
      const i4 v = *(const i4*)(smem_all + m * kWdPitch + c16 * 16);
      // nobody reads C again in this launch: keep it out of the way of A and B in L2
      __builtin_nontemporal_store(v, (i4*)(C + (size_t)(m0 + m) * p.N + kWdTileN * tn + c16 * 8));
    }
  }
  if (SLICED && threadIdx.x == 0) finish_leave(&p.locks[tile * p.lock_stride], ksplit);
}

template <bool GROUP, int RB>
static int configure_wide() {
  constexpr int lds = WdShape<RB>::kLdsBytes;
  return hipFuncSetAttribute((const void*)prefill_wide_kernel<GROUP, RB, false>,
                             hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess ||
         hipFuncSetAttribute((const void*)prefill_wide_kernel<GROUP, RB, true>,
                             hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess;
}
int configure_prefill_wide_kernels() {
  return configure_wide<false, 5>() | configure_wide<false, 6>() | configure_wide<false, 7>() |
                 configure_wide<false, 8>() | configure_wide<true, 5>() | configure_wide<true, 6>() |
                 configure_wide<true, 7>() | configure_wide<true, 8>()
             ? 3
             : 0;
}

template <bool GROUP, int RB>
static int launch_wide(const GemmArgs& a, int ksplit, hipStream_t stream) {
  constexpr int lds = WdShape<RB>::kLdsBytes;
  const int tiles_m = ceil_div(a.M, 16 * RB);
  const int tiles_n = a.N / kWdTileN;
  const dim3 grid(tiles_m * tiles_n * ksplit);
  if (ksplit > 1)
    hipLaunchKernelGGL((prefill_wide_kernel<GROUP, RB, true>), grid, dim3(256), lds, stream, a,
                       tiles_m, tiles_n, ksplit);
  else
    hipLaunchKernelGGL((prefill_wide_kernel<GROUP, RB, false>), grid, dim3(256), lds, stream, a,
                       tiles_m, tiles_n, 1);
  return launch_status();
}

int launch_prefill_wide(const GemmArgs& a, bool group, int tile_rows, int ksplit, hipStream_t stream) {
  switch (tile_rows + (group ? 1 : 0)) {
    case 80: return launch_wide<false, 5>(a, ksplit, stream);
    case 81: return launch_wide<true, 5>(a, ksplit, stream);
    case 96: return launch_wide<false, 6>(a, ksplit, stream);
    case 97: return launch_wide<true, 6>(a, ksplit, stream);
    case 112: return launch_wide<false, 7>(a, ksplit, stream);
    case 113: return launch_wide<true, 7>(a, ksplit, stream);
    case 128: return launch_wide<false, 8>(a, ksplit, stream);
    case 129: return launch_wide<true, 8>(a, ksplit, stream);
  }
  return 2;
}

}  // namespace w4a16
