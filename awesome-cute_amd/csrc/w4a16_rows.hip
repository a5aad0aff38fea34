// Column strips with up to 64 rows per workgroup: a workgroup owns CS 16-column
// strips (w4a16_strip.hip says what a strip is) and 16 MB rows over the whole k
// range.  For 17 rows and more, where a workgroup per 16 rows unpacks every weight
// several times, and a column tile that shares its k range among workgroups pays
// for their meeting (2 to 4 us of a launch of 10 to 15).
//
// What bounds it: what a compute unit takes in -- 32 MB k bytes of activations from the L2s
// beside 8 CS k bytes of weights.  Loads come back in order, so activations that the L2
// has (130 GB/s per compute unit by themselves) wait behind weights that it has not, and the
// two together come at the 57 to 61 GB/s that a compute unit draws from beyond its L2: M = 45,
// N = 12288, K = 4096 491 KB in 8 of 11.6 us.  Sets of strips and rows are chosen to keep
// both streams short (rows_plan in marlin_host.hip).
//
// Eight waves split the k range into contiguous runs of chunks of 64 k-values and
// meet once, at the end: no barrier in the loop, no scratch, no counters.  Activations
// and weights go straight to LDS (buffer_load ... lds), eight rows or lines of 128 bytes
// per load (four rows or fewer per load are 4 to 30 % slower), swizzled where they are
// fetched, and are read once in operand order.  MFMA lane (kg, nu) takes the sixteen
// k-values of row kg of four rows of B for column slot nu -- word j = (nu/2)%4 of the Marlin
// lanes (t, c = 2s + e), t = 0 ... 3, e = nu/8 -- so that an activation operand is eight
// neighbouring k-values of a row, 16 bytes.  (Weights through registers into LDS, and the
// scales of columns fetched after the loop, took 1.10 times as long: 528 problems over every
// pair but eight strips, 1.05 with five strips, 1.07 with six, 1.11 with two to four; 45 x 12288
// x 4096 13.0 us.)
//
// The more a wave has in flight the longer each takes to come: two chunks where strips and
// rows are few (a launch then waits for its first ones), else one, whose successor is
// requested before its arithmetic (M = 45, N = 12288, K = 4096: all weights requested at
// once 13.3 us, two units of 128 k-values 12.8, one 11.6; M = 18, N = 768, K = 2176, one
// strip and 16 rows, one chunk 0.90, two 0.85 and two units as well 0.82 of the time with
// weights through registers).  The last two chunks are steps of their own, which request
// nothing more.  (Requests past the end, dropped by the hardware's check, took as long as
// others: without them 0.97 of the time over 1128 problems, none more than 1.012, 0.93 where k
// is a chunk or two per wave.  11 x 16640 x 512 took 4.5 us with weights through registers, 5.15
// with requests past the end, 4.45 now.)
//
// Weights that only one workgroup reads are requested as read once, those of several row
// parts are not: two kernels.  (A branch on it in the loop took 1 % on average and 4 % with two
// strips, 16 rows and group scales.  As read once whatever the parts: 0.94 to 1.18 of the time
// over weights from memory, 2 to 12 % longer where a cache has them.)
//
// Eight strips are a kernel of their own (w4a16_rows_wide.hip).
#include "buffer_loads.hpp"
#include "w4a16_common.hpp"

namespace w4a16 {

namespace {

constexpr int kRowsWaves = 8;

// LDS accesses of the loop, outside the compiler's dependence tracking as well
template <int DW0, int DW1>  // offsets in dwords
__device__ __forceinline__ void rows_read2(unsigned at, i2& v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("ds_read2_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(v) : "v"(at), "n"(DW0), "n"(DW1) : "memory");
#endif
}

}  // namespace

// DEPTH chunks of activations in LDS per wave and UNITS units of weights: a unit is a chunk's,
// or with an odd number of strips those of two, which whole loads fetch
template <int CS, int MB, int DEPTH, int UNITS>
struct RowsShape {
  static constexpr int kALoads = 2 * MB;   // of 1 KiB per wave and chunk, eight rows
  static constexpr int kSlot = 2048 * MB;  // activations of a chunk
  static constexpr int kUnitChunks = CS % 2 == 0 ? 1 : 2;
  static constexpr int kBLoads = CS * kUnitChunks / 2;  // of 1 KiB, eight lines of 128 bytes
  static constexpr int kStagePerWave = DEPTH * kSlot + UNITS * 1024 * kBLoads;
  static_assert(UNITS == 1 || (UNITS == 2 && DEPTH == 2), "");
  // the waves' sums meet through LDS in passes of at most 16 blocks of 16 x 16
  static constexpr int kBlocks = CS * MB;
  static constexpr int kPasses = (kBlocks + 15) / 16;
  static constexpr int kPass = (kBlocks + kPasses - 1) / kPasses;
  static constexpr int kRounds = (kPass + kRowsWaves - 1) / kRowsWaves;  // blocks of a pass to a wave
  static constexpr int kReduce = kRowsWaves * kPass * 1024;
  static constexpr int kLds =
      kRowsWaves * kStagePerWave > kReduce ? kRowsWaves * kStagePerWave : kReduce;
};

// ONCE: the weights are requested as read once, where one workgroup reads them (launch_rows)
template <int CS, int MB, bool GROUP, int DEPTH, int UNITS, bool ONCE>
__global__ __launch_bounds__(64 * kRowsWaves) void rows_kernel(GemmArgs p) {
  using Sh = RowsShape<CS, MB, DEPTH, UNITS>;
  constexpr int NA = Sh::kALoads, NB = Sh::kBLoads, NS = GROUP ? CS : 0;
  extern __shared__ __attribute__((aligned(16))) char smem[];  // Sh::kLds
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int kg = lane >> 4;
  const int nu = lane & 15;
  // the parts of a strip set are neighbours behind one L2 (p.gpb carries the grid)
  const int wid = xcd_work_index((int)blockIdx.x, p.gpb);
  const int set = wid / p.row_parts;
  const int row0 = 16 * MB * (wid - set * p.row_parts);
  const int strip0 = set * CS;
  const int n_strips = p.N >> 4;  // (the last set may have fewer strips than CS)

  // my chunks [c0, c1): whole groups where there are groups, but no more than one chunk as long
  // as that keeps waves busy (16 rows, K = 512, four strips: four waves of two 1.14 times as long)
  const int chunks = p.K / 64;
  const bool pairs = GROUP && chunks > kRowsWaves;
  const int run = rows_run(wave);
  const int c0 = pairs ? 2 * (run * (chunks / 2) / kRowsWaves) : run * chunks / kRowsWaves;
  const int c1 = pairs ? 2 * ((run + 1) * (chunks / 2) / kRowsWaves) : (run + 1) * chunks / kRowsWaves;

  const __amdgpu_buffer_rsrc_t rB = make_rsrc(p.B, (unsigned)p.K * (unsigned)(p.N / 2));
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(p.A, (unsigned)p.M * (unsigned)p.K * 2u);
  const __amdgpu_buffer_rsrc_t rS =
      make_rsrc(p.S, (unsigned)(GROUP ? p.K / 128 : 1) * (unsigned)p.N * 2u);
  const int b_row = p.N * 8;  // bytes per row of B

  char* const stage = smem + wave * Sh::kStagePerWave;
  char* const stage_w = stage + DEPTH * Sh::kSlot;
  const unsigned lds_a = (unsigned)(size_t)stage, lds_w = lds_a + DEPTH * Sh::kSlot;
  // weights of a unit: its lines in the order [row][strip], eight lines per load.  Piece p
  // of a line sits at position p ^ (row % 4), which keeps the word reads (piece 4e + t of
  // four rows) from meeting in a bank.  The row is part of the offset that the hardware
  // checks: past the end of K there are zeros.
  int b_src[NB];
#pragma unroll
  for (int i = 0; i < NB; i++) {
    const int line = 8 * i + lane / 8, row = line / CS, strip = strip0 + line % CS;
    b_src[i] = strip < n_strips ? (4 * c0 + row) * b_row + 128 * strip + 16 * ((lane % 8) ^ (row & 3)) : kOob;
  }
  unsigned b_rd[4];
#pragma unroll
  for (int t = 0; t < 4; t++) b_rd[t] = lds_w + kg * CS * 128 + 64 * (nu >> 3) + 16 * (t ^ kg) + 4 * ((nu >> 1) & 3);
  const int shift = 8 * (nu & 1);  // h = nu%2 picks the low or the high byte pairs
  // activations: 128 bytes of eight rows per load; piece p of row r sits at position
  // p ^ (r % 8), so that the operand reads (piece 2 kg + q of row nu) meet no bank
  // twice.  Rows past M are zeros.
  int a_src[NA];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const int r = row0 + 8 * i + lane / 8;
    a_src[i] = r < p.M ? r * p.K * 2 + 16 * ((lane % 8) ^ (lane / 8)) : kOob;
  }
  unsigned a_rd[2];
#pragma unroll
  for (int q = 0; q < 2; q++) a_rd[q] = lds_a + nu * 128 + 16 * ((2 * kg + q) ^ (nu & 7));
  const int s_src = 2 * (16 * strip0 + nu);  // a group's scale of slot nu, 32 bytes per strip

  // One scale per column: those of the blocks that this wave writes in the end, in the
  // order of the passes (register r of lane (row, kg) holds slot 4 kg + r, column 16j +
  // 8h + 2s + e of the strip's block, e = kg / 2, j = 2 (kg % 2) + r / 2, h = r % 2)
  const int slot_col = 32 * (kg & 1) + (kg >> 1);
  unsigned short chan[Sh::kPasses][Sh::kRounds][4];
  if constexpr (!GROUP) {
#pragma unroll
    for (int ps = 0; ps < Sh::kPasses; ps++)
#pragma unroll
      for (int i = 0; i < Sh::kRounds; i++) {
        const int strip = strip0 + (ps * Sh::kPass + i * kRowsWaves + wave) / MB;
        const int col = 64 * (strip >> 2) + 2 * (strip & 3) + slot_col;
#pragma unroll
        for (int r = 0; r < 4; r++)  // (past the last column: zeros, and not used)
          chan[ps][i][r] = __builtin_amdgcn_raw_buffer_load_b16(
              rS, 2 * scale_index_single(col + 16 * (r >> 1) + 8 * (r & 1)), 0, 0);
      }
  }

  const DequantConsts dc;
  unsigned short sq[CS] = {}, sc[CS] = {};

  // What is not mine is requested at an offset past everything.
  auto issue_scales = [&](int c) {
    const int inv = c < c1 ? 0 : kOob;
#pragma unroll
    for (int s = 0; s < CS; s++)
      sq[s] = __builtin_amdgcn_raw_buffer_load_b16(rS, (s_src + 32 * s) | inv, (c >> 1) * p.N * 2, 0);
  };
  auto issue_rows = [&](int d, int c) {
    const int inv = c < c1 ? 0 : kOob;
#pragma unroll
    for (int i = 0; i < NA; i++) load_to_lds16(rA, stage + d * Sh::kSlot + 1024 * i, a_src[i] | inv, 128 * c);
  };
  // the unit that starts with chunk c, to place `at`
  auto issue_weights = [&](int at, int c) {
    const bool mine = c < c1;
    const int off = 4 * (c - c0) * b_row;
    char* const dst = stage_w + at * (1024 * NB);
#pragma unroll
    for (int i = 0; i < NB; i++) load_to_lds16<ONCE ? 2 : 0>(rB, dst + 1024 * i, mine ? b_src[i] + off : kOob, 0);
  };

  f4 acc[CS][MB];
#pragma unroll
  for (int s = 0; s < CS; s++)
#pragma unroll
    for (int m = 0; m < MB; m++) acc[s][m] = (f4){0.f, 0.f, 0.f, 0.f};

  const h2 sub = {(half_t)1032.f, (half_t)1032.f};
  const h2 mul = {(half_t)0.0625f, (half_t)0.0625f};
  const h2 add = {(half_t)-72.f, (half_t)-72.f};
  int w_at = 0;  // place of the unit in use
  // MORE: chunks follow c + 1.  Else c is the last or the last but one, and nothing is requested
  // that no step reads: the hardware takes as long over a request past the end as over another.
  auto step = [&](int c, auto EVEN, auto MORE) {
    constexpr bool even = decltype(EVEN)::value, more = decltype(MORE)::value;
    constexpr bool first = even || Sh::kUnitChunks == 1;                   // a unit of weights starts here
    constexpr bool last = !even || Sh::kUnitChunks == 1;                   // ... ends
    constexpr int d = DEPTH == 2 && !even ? 1 : 0;                         // this chunk's activations
    // chunk c has landed; what was requested after it may still be on its way (of the last two
    // chunks the second one's; the first of them may have come from before the loop)
    constexpr int later = DEPTH == 1 ? 0 : UNITS == 2 ? NA + NB + (even ? 0 : NS) : first ? NA : NS + NA;
    constexpr int later_of_two = DEPTH == 1 ? 0 : UNITS == 2 && Sh::kUnitChunks == 1 ? NA + NB : NA;
    __builtin_amdgcn_sched_barrier(0);
    if (more)
      __builtin_amdgcn_s_waitcnt(vmcnt(later));
    else if (even && later_of_two > 0 && c + 1 < c1)
      __builtin_amdgcn_s_waitcnt(vmcnt(later_of_two));
    else
      __builtin_amdgcn_s_waitcnt(vmcnt(0));
    __builtin_amdgcn_sched_barrier(0);
    i4 av[MB][2];
    for_each<MB>([&](auto I) {
      read_lds16<2048 * I.value>(a_rd[0] + d * Sh::kSlot, av[I.value][0]);
      read_lds16<2048 * I.value>(a_rd[1] + d * Sh::kSlot, av[I.value][1]);
    });
    // the four words of row kg, t = 0 ... 3, for every strip, two strips at a time
    constexpr int NP = (CS + 1) / 2;
    i2 wv[4][NP];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const unsigned at = b_rd[t] + w_at * (1024 * NB) + (first ? 0 : 512 * CS);
      for_each<NP>([&](auto I) {
        rows_read2<64 * I.value, 64 * I.value + (2 * I.value + 1 < CS ? 32 : 0)>(at, wv[t][I.value]);
      });
    }
    // every operand has come back: nothing stands between the reads and this, and
    // the registers are named so that they count as in use up to here
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(av[0][0]), "+v"(av[0][1]));
#pragma unroll
    for (int m = 1; m < MB; m++) asm volatile("" : "+v"(av[m][0]), "+v"(av[m][1]));
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int i = 0; i < NP; i++) asm volatile("" : "+v"(wv[t][i]));
#endif
    if (GROUP && even) {
#pragma unroll
      for (int s = 0; s < CS; s++) sc[s] = sq[s];
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (more) {
      if (GROUP && even) issue_scales(c + 2);
      __builtin_amdgcn_sched_barrier(0);
      // (two units: the rows first, so that a chunk's do not wait for later weights)
      if (UNITS == 2) issue_rows(d, c + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
      if (last) issue_weights(w_at, c + 1 + (UNITS - 1) * Sh::kUnitChunks);
      __builtin_amdgcn_sched_barrier(0);
      if (UNITS == 1) issue_rows(d, c + DEPTH);
    } else if (even && UNITS == 1 && c + 1 < c1) {
      if (last) issue_weights(w_at, c + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (DEPTH == 1) issue_rows(d, c + 1);
    }
    if (UNITS == 2 && last) w_at ^= 1;
    __builtin_amdgcn_sched_barrier(0);
    // a block of 16 slots: k-values 2t, 2t + 1 and 2t + 8, 2t + 9 of the lane's sixteen
#pragma unroll
    for (int s = 0; s < CS; s++) {
      h2 lo[4], hi[4];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const int w = (int)((unsigned)wv[t][s >> 1][s & 1] >> shift);
        lo[t] = as_h2((w & dc.lo_mask) | dc.ex) - sub;
        hi[t] = __builtin_elementwise_fma(as_h2((w & dc.hi_mask) | dc.ex), mul, add);
        if constexpr (GROUP) {
          const half_t x = __builtin_bit_cast(half_t, sc[s]);
          const h2 s2 = {x, x};
          lo[t] *= s2;
          hi[t] *= s2;
        }
      }
      const h8 w0 = make_h8(lo[0], lo[1], lo[2], lo[3]), w1 = make_h8(hi[0], hi[1], hi[2], hi[3]);
#pragma unroll
      for (int m = 0; m < MB; m++)
        acc[s][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w0, __builtin_bit_cast(h8, av[m][0]), acc[s][m], 0, 0, 0);
#pragma unroll
      for (int m = 0; m < MB; m++)
        acc[s][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w1, __builtin_bit_cast(h8, av[m][1]), acc[s][m], 0, 0, 0);
    }
  };

  if (GROUP) issue_scales(c0);
  __builtin_amdgcn_sched_barrier(0);
  issue_rows(0, c0);
  __builtin_amdgcn_sched_barrier(0);
  issue_weights(0, c0);
  __builtin_amdgcn_sched_barrier(0);
  if (DEPTH == 2 && c0 + 1 < c1) issue_rows(1, c0 + 1);
  __builtin_amdgcn_sched_barrier(0);
  if (UNITS == 2 && c0 + Sh::kUnitChunks < c1) issue_weights(1, c0 + Sh::kUnitChunks);
  int c = c0;
  for (; c + 2 < c1; c += 2) {
    step(c, std::true_type{}, std::true_type{});
    step(c + 1, std::false_type{}, std::true_type{});
  }
  if (c < c1) step(c, std::true_type{}, std::false_type{});
  if (c + 1 < c1) step(c + 1, std::false_type{}, std::false_type{});
  // nothing may still be on its way into LDS when it is reused
  __builtin_amdgcn_s_waitcnt(0);

  // ---- sum the eight waves, a block of 16 slots x 16 rows to a wave
  f4* const red = (f4*)smem;
#pragma unroll
  for (int ps = 0; ps < Sh::kPasses; ps++) {
    const int b0 = ps * Sh::kPass;
    __syncthreads();
#pragma unroll
    for (int b = b0; b < b0 + Sh::kPass && b < Sh::kBlocks; b++)
      red[(run * Sh::kPass + b - b0) * 64 + lane] = acc[b / MB][b % MB];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < Sh::kRounds; i++) {
      const int b = b0 + i * kRowsWaves + wave;
      if (b >= b0 + Sh::kPass || b >= Sh::kBlocks) continue;
      f4 v = red[(b - b0) * 64 + lane];
#pragma unroll
      for (int w = 1; w < kRowsWaves; w++) v += red[(w * Sh::kPass + b - b0) * 64 + lane];
      const int row = row0 + 16 * (b % MB) + nu;
      const int strip = strip0 + b / MB;
      if (strip >= n_strips) continue;
      // The lanes of both e, 32 apart, exchange halves and store two columns at a time.
      const int col = 64 * (strip >> 2) + 2 * (strip & 3) + 32 * (kg & 1);
      const int e = kg >> 1;
      unsigned o[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        half_t x = (half_t)v[r];
        if constexpr (!GROUP) x *= __builtin_bit_cast(half_t, chan[ps][i][r]);
        o[r] = __builtin_bit_cast(unsigned short, x);
      }
      const unsigned got = __shfl_xor((int)(e ? o[0] | (o[1] << 16) : o[2] | (o[3] << 16)), 32);
      if (row < p.M) {
        unsigned* const out = (unsigned*)((half_t*)p.C + (size_t)row * p.N + col + 16 * e);
        out[0] = e ? (got & 0xffffu) | (o[2] << 16) : o[0] | (got << 16);
        out[4] = e ? (got >> 16) | (o[3] << 16) : o[1] | (got & 0xffff0000u);
      }
    }
  }
}

namespace {

// calls f(kernel, LDS bytes) for a set of strips and rows that exists
template <class F>
bool with_rows_kernel(int strips, int blocks, bool group, bool once, F f) {
#define ROWS(CS, MB, DEPTH, UNITS, GROUP)                                               \
  if (strips == CS && blocks == MB && group == GROUP) {                               \
    using Sh = RowsShape<CS, MB, DEPTH, UNITS>;                                       \
    static_assert(Sh::kLds <= 160 * 1024, "LDS of a compute unit");                   \
    if (once)                                                                         \
      f(rows_kernel<CS, MB, GROUP, DEPTH, UNITS, true>, Sh::kLds);                    \
    else                                                                              \
      f(rows_kernel<CS, MB, GROUP, DEPTH, UNITS, false>, Sh::kLds);                   \
    return true;                                                                      \
  }
#define ROWS_OF_BOTH(CS, MB, DEPTH, UNITS) ROWS(CS, MB, DEPTH, UNITS, true) ROWS(CS, MB, DEPTH, UNITS, false)
  ROWS_OF_BOTH(1, 1, 2, 2)
  ROWS_OF_BOTH(2, 1, 2, 2)
  ROWS_OF_BOTH(3, 1, 2, 1)
  ROWS_OF_BOTH(4, 1, 2, 1)
  ROWS_OF_BOTH(2, 2, 2, 2)
  ROWS_OF_BOTH(3, 2, 1, 1)
  ROWS_OF_BOTH(4, 2, 1, 1)
  ROWS_OF_BOTH(6, 2, 1, 1)
  ROWS_OF_BOTH(2, 3, 1, 1)
  ROWS_OF_BOTH(3, 3, 1, 1)
  ROWS_OF_BOTH(4, 3, 1, 1)
  ROWS_OF_BOTH(5, 3, 1, 1)
  ROWS_OF_BOTH(6, 3, 1, 1)
  ROWS(4, 4, 1, 1, true)
  ROWS_OF_BOTH(5, 4, 1, 1)
  ROWS_OF_BOTH(6, 4, 1, 1)
#undef ROWS_OF_BOTH
#undef ROWS
  return false;
}

}  // namespace

bool rows_exist(int strips, int blocks, bool group) {
  return strips == 8 ? rows_wide_exist(blocks) : with_rows_kernel(strips, blocks, group, true, [](auto, int) {});
}

int configure_rows_kernels() {
  bool ok = true;
  for (int strips = 1; strips <= kRowsMaxStrips; strips++)
    for (int blocks = 1; blocks <= kRowsMaxBlocks; blocks++)
      for (const bool group : {false, true})
        for (const bool once : {false, true})
          with_rows_kernel(strips, blocks, group, once, [&](auto kernel, int lds) {
            ok = ok && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           lds) == hipSuccess;
          });
  return ok ? 0 : 3;
}

int launch_rows(const GemmArgs& a, bool group, int strips, int blocks, hipStream_t stream) {
  if (strips == 8) return launch_rows_wide(a, group, blocks, stream);
  GemmArgs b = a;
  b.row_parts = ceil_div(a.M, 16 * blocks);
  b.gpb = ceil_div(a.N / 16, strips) * b.row_parts;
  const bool found = with_rows_kernel(strips, blocks, group, b.row_parts == 1, [&](auto kernel, int lds) {
    hipLaunchKernelGGL(kernel, dim3(b.gpb), dim3(64 * kRowsWaves), lds, stream, b);
  });
  return found ? launch_status() : 2;
}

}  // namespace w4a16
