// The rows kernel (w4a16_rows.hip says what it is for) over eight strips: two whole
// 64-column blocks and 16 MB <= 64 rows per workgroup, over the whole k range.
//
// A lane takes its 16-byte pieces (t = kg, c = nu%8) of four rows of B straight into
// registers, and four lane swaps per four words turn rows into lane groups -- no LDS for
// the weights.  That is what many columns and 33 rows and more take (M = 64, N = 28672, K =
// 8192, in turn on one box: 44.6 us on 64-row prefill tiles, 42.9 so; on others 42.6 and
// 41.7, 49.4 and 41.6; with seven strips through LDS 45.5).
//
// Bound: what the compute unit takes in.  1.5 MB each at M = 64, N = 28672, K = 8192, two
// thirds of them activations, in a loop of 27 us: 57 GB/s, as much as a compute unit draws
// from beyond its L2.  Its loads come back in order, so activations that the L2 has wait
// behind weights that it has not: in builds without the rest the loop takes 28 us for the
// loads alone, 15 for the weights', 10 for the activations', 23 for the arithmetic (whole
// launches 35.4, 23.7, 16.3 and 29.5).
//
// rows_deep_kernel, for 33 rows and more over a deep k: weights requested three chunks ahead,
// activations two, and the unpack dealt out behind the MFMAs of the operand before
// (gen_rows_wide.py).  Its start and its code are longer.  Time by it over the time
// without, means over 1435 problems of one to four row parts by k in steps of 512, four row
// blocks: from k = 2560 0.996, 3072 0.989, 3584 0.985, 4096 0.978, 5120 0.967, 6656 0.964;
// three: 1.029, 1.018, 1.010, 1.005, from 4608 0.999, 5120 0.994, 6656 0.989; 64 x 28672 x
// 8192 42.1 -> 41.2 us.
#include "buffer_loads.hpp"
#include "w4a16_common.hpp"

namespace w4a16 {

namespace {

constexpr int kWaves = 8;
constexpr int kDeepLds = kWaves * 2 * 8192;  // rows_deep_kernel: two slots per wave

template <int MB>
struct WideShape {
  static constexpr int kSlot = 2048 * MB;             // activations of a chunk
  static constexpr int kPasses = (8 * MB + 15) / 16;  // the waves' sums meet in passes of at most 16 blocks
  static constexpr int kPass = 8 * MB / kPasses;
  static constexpr int kRounds = (kPass + kWaves - 1) / kWaves;  // blocks of a pass to a wave
  static constexpr int kReduce = kWaves * kPass * 1024;
  static constexpr int kLds = kWaves * kSlot > kReduce ? kWaves * kSlot : kReduce;
};

// the waves' sums meet, a block of 16 slots x 16 rows to a wave, and C is written
template <int MB, bool GROUP>
__device__ __forceinline__ void wide_finish(const GemmArgs& p, char* smem, const f4 (&acc)[8][MB],
                                            const __amdgpu_buffer_rsrc_t rS, int set, int row0, int wave, int lane) {
  using Sh = WideShape<MB>;
  const int kg = lane >> 4, nu = lane & 15;
  f4* const red = (f4*)smem;
#pragma unroll
  for (int ps = 0; ps < Sh::kPasses; ps++) {
    const int b0 = ps * Sh::kPass;
    // (one scale per column: on their way while the sums meet)
    h4 chan[Sh::kRounds];
    const int col0 = 128 * set + 64 * (kg >> 1) + 4 * (kg & 1);
    if constexpr (!GROUP) {
#pragma unroll
      for (int i = 0; i < Sh::kRounds; i++) {
        const int s = (b0 + i * kWaves + wave) / MB;
#pragma unroll
        for (int r = 0; r < 4; r++)
          chan[i][r] = __builtin_bit_cast(
              half_t, __builtin_amdgcn_raw_buffer_load_b16(
                          rS, 2 * scale_index_single(col0 + 16 * (s >> 1) + 8 * (s & 1) + r), 0, 0));
      }
    }
    __syncthreads();
#pragma unroll
    for (int b = b0; b < b0 + Sh::kPass; b++) red[(rows_run(wave) * Sh::kPass + b - b0) * 64 + lane] = acc[b / MB][b % MB];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < Sh::kRounds; i++) {
      const int b = b0 + i * kWaves + wave;
      if (b >= b0 + Sh::kPass) continue;
      f4 v = red[(b - b0) * 64 + lane];
#pragma unroll
      for (int w = 1; w < kWaves; w++) v += red[(w * Sh::kPass + b - b0) * 64 + lane];
      const int row = row0 + 16 * (b % MB) + nu;
      // register r of lane (row, kg) holds column slot nu' = 4 kg + r, column 16j +
      // 8h + nu' % 8 of block nu' / 8, b / MB = 2j + h: four neighbouring columns
      const int s = b / MB;
      const int col = col0 + 16 * (s >> 1) + 8 * (s & 1);
      h4 o = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
      if constexpr (!GROUP) o *= chan[i];
      if (row < p.M) *(h4*)((half_t*)p.C + (size_t)row * p.N + col) = o;
    }
  }
}

// what a lane of either kernel computes and where its pieces lie
template <int MB, bool GROUP>
struct WideLane {
  int wave, lane, kg, nu;
  int set, row0;  // my strip set, my first row
  int c0, c1;     // my chunks of 64 k-values: whole groups where there are groups
  // this lane's 16-byte pieces of B (Marlin lane t = kg, c = nu%8 of block nu/8) and, of a
  // group, the scales of columns 16j + 8h + c of that block
  int b_src, s_src;
  // activations: 128 bytes of eight rows per load; piece p of row r sits at position p ^ (r % 8),
  // so that the operand reads (piece 2 kg + q of row nu) meet no bank twice.  Rows past M are
  // zeros.
  int a_src[2 * MB];

  __device__ __forceinline__ explicit WideLane(const GemmArgs& p) {
    const int tid = threadIdx.x;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    lane = tid & 63;
    kg = lane >> 4;
    nu = lane & 15;
    // the parts of a strip set are neighbours behind one L2 (p.gpb carries the grid)
    const int wid = xcd_work_index((int)blockIdx.x, p.gpb);
    set = wid / p.row_parts;
    row0 = 16 * MB * (wid - set * p.row_parts);
    const int chunks = p.K / 64;
    const int run = rows_run(wave);
    c0 = GROUP ? 2 * (run * (chunks / 2) / kWaves) : run * chunks / kWaves;
    c1 = GROUP ? 2 * ((run + 1) * (chunks / 2) / kWaves) : (run + 1) * chunks / kWaves;
    b_src = 1024 * set + 512 * (nu >> 3) + 16 * (4 * (nu & 7) + kg);
    s_src = 256 * set + 128 * (nu >> 3) + 16 * (nu & 7);
#pragma unroll
    for (int i = 0; i < 2 * MB; i++) {
      const int r = row0 + 8 * i + lane / 8;
      a_src[i] = r < p.M ? r * p.K * 2 + 16 * ((lane % 8) ^ (lane / 8)) : kOob;
    }
  }
  __device__ __forceinline__ unsigned a_rd(int q) const { return nu * 128 + 16 * ((2 * kg + q) ^ (nu & 7)); }
};

}  // namespace

template <int MB, bool GROUP>
__global__ __launch_bounds__(64 * kWaves) void rows_wide_kernel(GemmArgs p) {
  using Sh = WideShape<MB>;
  constexpr int NA = 2 * MB;
  extern __shared__ __attribute__((aligned(16))) char smem[];  // Sh::kLds
  const WideLane<MB, GROUP> me(p);

  const __amdgpu_buffer_rsrc_t rB = make_rsrc(p.B, (unsigned)p.K * (unsigned)(p.N / 2));
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(p.A, (unsigned)p.M * (unsigned)p.K * 2u);
  const __amdgpu_buffer_rsrc_t rS =
      make_rsrc(p.S, (unsigned)(GROUP ? p.K / 128 : 1) * (unsigned)p.N * 2u);
  const int b_row = p.N * 8;  // bytes per row of B

  char* const stage = smem + me.wave * Sh::kSlot;
  const unsigned lds_a = (unsigned)(size_t)stage;
  const unsigned a_rd[2] = {lds_a + me.a_rd(0), lds_a + me.a_rd(1)};

  const DequantConsts dc;
  i4 bq[4];
  i4 sq = {}, sc = {};

  // Request chunk c, and with an even one the scales of its group; a chunk that is not
  // mine is requested at an offset past everything.
  auto issue = [&](int c, bool even) {
    __builtin_amdgcn_sched_barrier(0);
    const int inv = c < me.c1 ? 0 : kOob;
    if (GROUP && even) sq = __builtin_amdgcn_raw_buffer_load_b128(rS, me.s_src | inv, (c >> 1) * p.N * 2, 0);
#pragma unroll
    for (int i = 0; i < 4; i++)
      bq[i] = __builtin_amdgcn_raw_buffer_load_b128(rB, me.b_src | inv, (4 * c + i) * b_row, 2);
#pragma unroll
    for (int i = 0; i < NA; i++) load_to_lds16(rA, stage + 1024 * i, me.a_src[i] | inv, 128 * c);
    __builtin_amdgcn_sched_barrier(0);
  };

  f4 acc[8][MB];
#pragma unroll
  for (int s = 0; s < 8; s++)
#pragma unroll
    for (int m = 0; m < MB; m++) acc[s][m] = (f4){0.f, 0.f, 0.f, 0.f};

  auto step = [&](int c, auto EVEN) {
    constexpr bool even = decltype(EVEN)::value;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(vmcnt(0));  // chunk c has landed
    __builtin_amdgcn_sched_barrier(0);
    i4 av[MB][2];
    for_each<MB>([&](auto I) {
      read_lds16<2048 * I.value>(a_rd[0], av[I.value][0]);
      read_lds16<2048 * I.value>(a_rd[1], av[I.value][1]);
    });
    // the words of row kg, t = 0 ... 3, for every j, a word holding columns 16j + c and
    // 16j + 8 + c
    i2 wv[4][2];
    // every operand has come back: nothing stands between the reads and this, and
    // the registers are named so that they count as in use up to here
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(av[0][0]), "+v"(av[0][1]));
#pragma unroll
    for (int m = 1; m < MB; m++) asm volatile("" : "+v"(av[m][0]), "+v"(av[m][1]));
    // lane group t of register i holds row i: a 4 x 4 transpose over the two
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const auto x = __builtin_amdgcn_permlane32_swap(bq[0][j], bq[2][j], false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(bq[1][j], bq[3][j], false, false);
      const auto u = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
      const auto v = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
      wv[j][0] = (i2){(int)u[0], (int)u[1]};
      wv[j][1] = (i2){(int)v[0], (int)v[1]};
    }
#endif
    if (GROUP && even) sc = sq;
    issue(c + 1, !even);
    // a block of 16 slots: k-values 2t, 2t + 1 and 2t + 8, 2t + 9 of the lane's sixteen
    const auto multiply = [&](const h2(&lo)[4], const h2(&hi)[4], f4(&sum)[MB]) {
      const h8 w0 = make_h8(lo[0], lo[1], lo[2], lo[3]), w1 = make_h8(hi[0], hi[1], hi[2], hi[3]);
#pragma unroll
      for (int m = 0; m < MB; m++)
        sum[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w0, __builtin_bit_cast(h8, av[m][0]), sum[m], 0, 0, 0);
#pragma unroll
      for (int m = 0; m < MB; m++)
        sum[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w1, __builtin_bit_cast(h8, av[m][1]), sum[m], 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < 4; j++) {
      h2 lo[4], hi[4], lo8[4], hi8[4];  // (of column c + 8)
#pragma unroll
      for (int t = 0; t < 4; t++)
        dequant_word<GROUP>(wv[j][t >> 1][t & 1], as_h2(sc[j]), dc, lo[t], hi[t], lo8[t], hi8[t]);
      multiply(lo, hi, acc[2 * j]);
      multiply(lo8, hi8, acc[2 * j + 1]);
    }
  };

  issue(me.c0, true);
  for (int c = me.c0; c < me.c1; c += 2) {
    step(c, std::true_type{});
    if (c + 1 < me.c1) step(c + 1, std::false_type{});
  }
  // nothing may still be on its way into LDS when it is reused
  __builtin_amdgcn_s_waitcnt(0);

  wide_finish<MB, GROUP>(p, smem, acc, rS, me.set, me.row0, me.wave, me.lane);
}

// The same over a deep k range, with the loop that gen_rows_wide.py writes: weights requested
// three chunks ahead, activations two.
template <int MB, bool GROUP>
__global__ __launch_bounds__(64 * kWaves) void rows_deep_kernel(GemmArgs p) {
  constexpr int kSlot = 8192;  // activations of a chunk, slots swapped by an exclusive or
  extern __shared__ __attribute__((aligned(16))) char smem[];  // kDeepLds
  const WideLane<MB, GROUP> me(p);

  i4 rb_words = rsrc_words(p.B, (unsigned)p.K * (unsigned)(p.N / 2));
  i4 ra_words = rsrc_words(p.A, (unsigned)p.M * (unsigned)p.K * 2u);
  i4 rs_words = rsrc_words(p.S, (unsigned)(GROUP ? p.K / 128 : 1) * (unsigned)p.N * 2u);
  const int b_row = p.N * 8;  // bytes per row of B
  const int s_row = p.N * 2;
  const int b_src = me.b_src, s_src = me.s_src, c0 = me.c0, c1 = me.c1;
  const int(&a_src)[2 * MB] = me.a_src;
  unsigned lds_slot = (unsigned)(size_t)smem + me.wave * 2 * kSlot;  // (the only LDS of the kernel: at 0)
  unsigned a_rd[2] = {lds_slot + me.a_rd(0), lds_slot + me.a_rd(1)};

  f4 acc[8][MB];
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(MB == 3 || MB == 4, "");
  if constexpr (GROUP && MB == 4) {
#include "w4a16_rows_wide_group64.inc"
  } else if constexpr (GROUP && MB == 3) {
#include "w4a16_rows_wide_group48.inc"
  } else if constexpr (MB == 4) {
#include "w4a16_rows_wide_chan64.inc"
  } else {
#include "w4a16_rows_wide_chan48.inc"
  }
#else  // the host pass only needs the launch stub
  (void)rb_words, (void)ra_words, (void)rs_words, (void)b_row, (void)s_row, (void)b_src, (void)s_src;
  (void)a_src, (void)a_rd, (void)lds_slot, (void)c0, (void)c1;
  for (auto& r : acc)
    for (auto& v : r) v = (f4){0.f, 0.f, 0.f, 0.f};
#endif

  __amdgpu_buffer_rsrc_t rS = make_rsrc(p.S, (unsigned)(GROUP ? p.K / 128 : 1) * (unsigned)p.N * 2u);
  // (the lane once more, so that no register is held through the statement, which leaves six)
  const int again = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0));
  wide_finish<MB, GROUP>(p, smem, acc, rS, me.set, me.row0, me.wave, again);
}

namespace {

template <class F>
bool with_wide_kernel(int blocks, bool group, bool deep, F f) {
  switch ((deep ? 100 : 0) + 2 * blocks + (group ? 1 : 0)) {
    case 106: f(rows_deep_kernel<3, false>, kDeepLds); return true;
    case 107: f(rows_deep_kernel<3, true>, kDeepLds); return true;
    case 108: f(rows_deep_kernel<4, false>, kDeepLds); return true;
    case 109: f(rows_deep_kernel<4, true>, kDeepLds); return true;
    case 4: f(rows_wide_kernel<2, false>, WideShape<2>::kLds); return true;
    case 5: f(rows_wide_kernel<2, true>, WideShape<2>::kLds); return true;
    case 6: f(rows_wide_kernel<3, false>, WideShape<3>::kLds); return true;
    case 7: f(rows_wide_kernel<3, true>, WideShape<3>::kLds); return true;
    case 8: f(rows_wide_kernel<4, false>, WideShape<4>::kLds); return true;
    case 9: f(rows_wide_kernel<4, true>, WideShape<4>::kLds); return true;
  }
  return false;
}

}  // namespace

bool rows_wide_exist(int blocks) {
  return with_wide_kernel(blocks, true, false, [](auto, int) {});
}

int configure_rows_wide_kernels() {
  bool ok = true;
  for (int blocks = 1; blocks <= kRowsMaxBlocks; blocks++)
    for (const bool group : {false, true})
      for (const bool deep : {false, true})
        with_wide_kernel(blocks, group, deep, [&](auto kernel, int lds) {
          ok = ok && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         lds) == hipSuccess;
        });
  return ok ? 0 : 3;
}

int launch_rows_wide(const GemmArgs& a, bool group, int blocks, hipStream_t stream) {
  if (a.N % 128 != 0) return 2;
  GemmArgs b = a;
  b.row_parts = ceil_div(a.M, 16 * blocks);
  b.gpb = a.N / 128 * b.row_parts;
  // (from where it is a hundredth faster with four row blocks, half that with three)
  const bool deep = (blocks == 4 && a.K >= 3072) || (blocks == 3 && a.K >= 5120);
  const bool found = with_wide_kernel(blocks, group, deep, [&](auto kernel, int lds) {
    hipLaunchKernelGGL(kernel, dim3(b.gpb), dim3(64 * kWaves), lds, stream, b);
  });
  return found ? launch_status() : 2;
}

}  // namespace w4a16
