// Column strips with up to 64 rows per workgroup: a workgroup owns CS 16-column
// strips (w4a16_strip.hip says what a strip is) and 16 MB rows over the whole k
// range.  For 17 rows and more, where a workgroup per 16 rows unpacks every weight
// several times, and a column tile that shares its k range among workgroups pays
// for their meeting (2 to 4 us of a launch of 10 to 15).
//
// What bounds it: what a compute unit takes in, 55 to 60 GB/s with all of them at
// work -- 32 MB k bytes of activations from the L2s beside 8 CS k bytes of weights
// -- and what its LDS takes in, 64 bytes per clock whatever the width of the stores
// (reads come at 230).  So the activations go straight to LDS (buffer_load ... lds)
// and are read once, as whole operands: sets of strips and rows are chosen to keep
// both streams short (rows_plan in marlin_host.hip).  M = 45, N = 12288, K = 4096:
// 15.1 us streaming, 12.7 so; M = 46, N = 18432, K = 4480 29.2 and 18.4.
//
// Eight waves split the k range into contiguous runs of chunks of 64 k-values and
// meet once, at the end: no barrier in the loop, no scratch, no counters.  The
// weights of a chunk are fetched 16 bytes per lane, four rows of B, and pass
// through LDS into operand order.  MFMA lane (kg, nu) takes the sixteen k-values of
// row kg of the four for column slot nu -- word j = (nu/2)%4 of the Marlin lanes
// (t, c = 2s + e), t = 0 ... 3, e = nu/8 -- so that an activation operand is eight
// neighbouring k-values of a row, 16 bytes.
//
// Eight strips are two whole 64-column blocks: a lane then takes its 16-byte pieces
// (t = kg, c = nu%8) of four rows of B straight into registers, and four lane swaps
// per four words turn rows into lane groups -- no LDS for the weights.  That is
// what many columns and 33 rows and more take (M = 64, N = 28672, K = 8192, in turn on
// one box: 44.6 us on 64-row prefill tiles, 42.9 so; on others 42.6 and 41.7, 49.4 and
// 41.6; with seven strips through LDS 45.5).  Neither the matrix units (busy 42 % of the
// cycles) nor the issue of vector operations (57 %) is full there: a chunk's loads are
// requested before the arithmetic of the one before it and waited for after it, and
// the two take turns; without loads the launch takes two thirds of its time.
//
// The more chunks a wave has in flight the longer each takes to come: two where
// strips and rows are few (a launch then waits for its first ones), else one, whose
// successor is requested before its arithmetic (M = 45, N = 12288, K = 4096: one
// 12.9 us, two 13.6; M = 111, N = 512, K = 4992, one strip and 16
// rows: two 6.6 us).
#include <type_traits>

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
__device__ __forceinline__ void rows_write16(unsigned at, i4 v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("ds_write_b128 %0, %1" ::"v"(at), "v"(v) : "memory");
#endif
}

template <int N, class F>
__device__ __forceinline__ void rows_each(F f) {
  if constexpr (N > 0) {
    rows_each<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

}  // namespace

template <int CS, int MB, int DEPTH>
struct RowsShape {
  static constexpr bool kWide = CS == 8;
  static constexpr int kBLoads = (CS + 1) / 2;  // of 1 KiB per wave and chunk, eight lines of 128 bytes
  static constexpr int kALoads = 2 * MB;        // ... eight rows
  static constexpr int kSlot = 2048 * MB;       // activations of a chunk
  static constexpr int kBRow = CS * 128 + 16;   // a row of B in LDS
  static constexpr int kStagePerWave = DEPTH * kSlot + (kWide ? 0 : 4 * kBRow);
  // the waves' sums meet through LDS in passes of at most 16 blocks of 16 x 16
  static constexpr int kBlocks = CS * MB;
  static constexpr int kPasses = (kBlocks + 15) / 16;
  static constexpr int kPass = (kBlocks + kPasses - 1) / kPasses;
  static constexpr int kReduce = kRowsWaves * kPass * 1024;
  static constexpr int kLds =
      kRowsWaves * kStagePerWave > kReduce ? kRowsWaves * kStagePerWave : kReduce;
  static_assert(kLds <= 160 * 1024, "LDS of a compute unit");
  static_assert(!kWide || DEPTH == 1, "its weights are taken from one slot");
};

template <int CS, int MB, bool GROUP, int DEPTH>
__global__ __launch_bounds__(64 * kRowsWaves) void rows_kernel(GemmArgs p) {
  using Sh = RowsShape<CS, MB, DEPTH>;
  constexpr int NA = Sh::kALoads, NB = Sh::kBLoads;
  constexpr bool WIDE = Sh::kWide;
  constexpr int NS = !GROUP ? 0 : WIDE ? 1 : CS;  // scale loads per group
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

  // my chunks [c0, c1): whole groups where there are groups
  const int chunks = p.K / 64;
  const int c0 = GROUP ? 2 * (wave * (chunks / 2) / kRowsWaves) : wave * chunks / kRowsWaves;
  const int c1 = GROUP ? 2 * ((wave + 1) * (chunks / 2) / kRowsWaves) : (wave + 1) * chunks / kRowsWaves;

  const __amdgpu_buffer_rsrc_t rB = make_rsrc(p.B, (unsigned)p.K * (unsigned)(p.N / 2));
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(p.A, (unsigned)p.M * (unsigned)p.K * 2u);
  const __amdgpu_buffer_rsrc_t rS =
      make_rsrc(p.S, (unsigned)(GROUP ? p.K / 128 : 1) * (unsigned)p.N * 2u);
  const int b_row = p.N * 8;  // bytes per row of B

  char* const stage = smem + wave * Sh::kStagePerWave;
  const unsigned lds_a = (unsigned)(size_t)stage, lds_b = lds_a + DEPTH * Sh::kSlot;
  // weights: lines in the order [row][strip]; lanes past the last line fetch
  // nothing and write to the padding.  Eight strips: pieces of one row per load.
  int b_src[WIDE ? 1 : NB];
  unsigned b_wr[NB];
  if constexpr (WIDE) {
    b_src[0] = 128 * strip0 + 512 * (nu >> 3) + 16 * (4 * (nu & 7) + kg);
  } else {
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int line = 8 * i + lane / 8, row = line / CS, strip = strip0 + line % CS;
      const bool on = line < 4 * CS;
      b_src[i] = on && strip < n_strips ? row * b_row + 128 * strip + 16 * (lane % 8) : kOob;
      b_wr[i] = lds_b + (on ? row * Sh::kBRow + 128 * (line % CS) + 16 * (lane % 8) : 3 * Sh::kBRow + CS * 128);
    }
  }
  const unsigned b_rd = lds_b + kg * Sh::kBRow + 64 * (nu >> 3) + 4 * ((nu >> 1) & 3);
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
  // a group's scale of slot nu, 32 bytes per strip; eight strips: those of columns
  // 16j + 8h + c of my block, in one 16-byte piece
  const int s_src = WIDE ? 32 * strip0 + 128 * (nu >> 3) + 16 * (nu & 7) : 2 * (16 * strip0 + nu);

  const DequantConsts dc;
  i4 bq[DEPTH][NB];
  using Scales = std::conditional_t<WIDE, i4, unsigned short[CS]>;
  Scales sq = {}, sc = {};

  // Request chunk c into slot d, and with an even one the scales of its group; a
  // chunk that is not mine is requested at an offset past everything.
  auto issue = [&](int d, int c, bool even) {
    __builtin_amdgcn_sched_barrier(0);
    const int inv = c < c1 ? 0 : kOob;
    if (GROUP && even) {
      if constexpr (WIDE) {
        sq = __builtin_amdgcn_raw_buffer_load_b128(rS, s_src | inv, (c >> 1) * p.N * 2, 0);
      } else {
#pragma unroll
        for (int s = 0; s < CS; s++)
          sq[s] = __builtin_amdgcn_raw_buffer_load_b16(rS, (s_src + 32 * s) | inv, (c >> 1) * p.N * 2, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < NB; i++)
      bq[d][i] = __builtin_amdgcn_raw_buffer_load_b128(rB, b_src[WIDE ? 0 : i] | inv,
                                                       (WIDE ? 4 * c + i : 4 * c) * b_row, 2);
#pragma unroll
    for (int i = 0; i < NA; i++) load_to_lds16(rA, stage + d * Sh::kSlot + 1024 * i, a_src[i] | inv, 128 * c);
    __builtin_amdgcn_sched_barrier(0);
  };

  f4 acc[CS][MB];
#pragma unroll
  for (int s = 0; s < CS; s++)
#pragma unroll
    for (int m = 0; m < MB; m++) acc[s][m] = (f4){0.f, 0.f, 0.f, 0.f};

  const h2 sub = {(half_t)1032.f, (half_t)1032.f};
  const h2 mul = {(half_t)0.0625f, (half_t)0.0625f};
  const h2 add = {(half_t)-72.f, (half_t)-72.f};
  auto step = [&](int d, int c, auto EVEN) {
    constexpr bool even = decltype(EVEN)::value;
    // chunk c has landed; the one after it may still be on its way
    constexpr int later = DEPTH == 1 ? 0 : NA + NB + (even ? 0 : NS);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(vmcnt(later));
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!WIDE) {
#pragma unroll
      for (int i = 0; i < NB; i++) rows_write16(b_wr[i], bq[d][i]);
    }
    i4 av[MB][2];
    const unsigned slot = d * Sh::kSlot;
    rows_each<MB>([&](auto I) {
      read_lds16<2048 * I.value>(a_rd[0] + slot, av[I.value][0]);
      read_lds16<2048 * I.value>(a_rd[1] + slot, av[I.value][1]);
    });
    // the four words of row kg, t = 0 ... 3, for every strip (eight strips: for every j,
    // a word holding columns 16j + c and 16j + 8 + c)
    constexpr int NW = WIDE ? 4 : CS;
    i2 wv[NW][2];
    if constexpr (!WIDE)
      rows_each<CS>([&](auto I) {
        rows_read2<32 * I.value, 32 * I.value + 4>(b_rd, wv[I.value][0]);
        rows_read2<32 * I.value + 8, 32 * I.value + 12>(b_rd, wv[I.value][1]);
      });
    // every operand has come back: nothing stands between the reads and this, and
    // the registers are named so that they count as in use up to here
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(av[0][0]), "+v"(av[0][1]));
#pragma unroll
    for (int m = 1; m < MB; m++) asm volatile("" : "+v"(av[m][0]), "+v"(av[m][1]));
    if constexpr (!WIDE) {
#pragma unroll
      for (int s = 0; s < CS; s++) asm volatile("" : "+v"(wv[s][0]), "+v"(wv[s][1]));
    } else {
      // lane group t of register i holds row i: a 4 x 4 transpose over the two
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const auto x = __builtin_amdgcn_permlane32_swap(bq[d][0][j], bq[d][2][j], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(bq[d][1][j], bq[d][3][j], false, false);
        const auto u = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
        const auto v = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
        wv[j][0] = (i2){(int)u[0], (int)u[1]};
        wv[j][1] = (i2){(int)v[0], (int)v[1]};
      }
    }
#endif
    if (GROUP && even) {
      if constexpr (WIDE) {
        sc = sq;
      } else {
#pragma unroll
        for (int s = 0; s < CS; s++) sc[s] = sq[s];
      }
    }
    issue(d, c + DEPTH, DEPTH == 1 ? !even : even);
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
    for (int s = 0; s < NW; s++) {
      h2 lo[4], hi[4];
      if constexpr (WIDE) {
        h2 lo8[4], hi8[4];  // of column c + 8
#pragma unroll
        for (int t = 0; t < 4; t++)
          dequant_word<GROUP>(wv[s][t >> 1][t & 1], as_h2(sc[s]), dc, lo[t], hi[t], lo8[t], hi8[t]);
        multiply(lo, hi, acc[2 * s]);
        multiply(lo8, hi8, acc[2 * s + 1]);
      } else {
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const int w = (int)((unsigned)wv[s][t >> 1][t & 1] >> shift);
          lo[t] = as_h2((w & dc.lo_mask) | dc.ex) - sub;
          hi[t] = __builtin_elementwise_fma(as_h2((w & dc.hi_mask) | dc.ex), mul, add);
          if constexpr (GROUP) {
            const half_t x = __builtin_bit_cast(half_t, sc[s]);
            const h2 s2 = {x, x};
            lo[t] *= s2;
            hi[t] *= s2;
          }
        }
        multiply(lo, hi, acc[s]);
      }
    }
  };

#pragma unroll
  for (int d = 0; d < DEPTH; d++) issue(d, c0 + d, d == 0);
  for (int c = c0; c < c1; c += 2) {
    step(0, c, std::true_type{});
    if (c + 1 < c1) step(DEPTH - 1, c + 1, std::false_type{});
  }
  // nothing may still be on its way into LDS when it is reused
  __builtin_amdgcn_s_waitcnt(0);

  // ---- sum the eight waves, a block of 16 slots x 16 rows to a wave
  f4* const red = (f4*)smem;
#pragma unroll
  for (int b0 = 0; b0 < Sh::kBlocks; b0 += Sh::kPass) {
    __syncthreads();
#pragma unroll
    for (int b = b0; b < b0 + Sh::kPass && b < Sh::kBlocks; b++)
      red[(wave * Sh::kPass + b - b0) * 64 + lane] = acc[b / MB][b % MB];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (Sh::kPass + kRowsWaves - 1) / kRowsWaves; i++) {
      const int b = b0 + i * kRowsWaves + wave;
      if (b >= b0 + Sh::kPass || b >= Sh::kBlocks) continue;
      f4 v = red[(b - b0) * 64 + lane];
#pragma unroll
      for (int w = 1; w < kRowsWaves; w++) v += red[(w * Sh::kPass + b - b0) * 64 + lane];
      const int row = row0 + 16 * (b % MB) + nu;
      if constexpr (WIDE) {
        // register r of lane (row, kg) holds column slot nu' = 4 kg + r, column 16j +
        // 8h + nu' % 8 of block nu' / 8, b / MB = 2j + h: four neighbouring columns
        const int s = b / MB;
        const int col = 16 * strip0 + 64 * (kg >> 1) + 16 * (s >> 1) + 8 * (s & 1) + 4 * (kg & 1);
        h4 o = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
        if constexpr (!GROUP) {
#pragma unroll
          for (int r = 0; r < 4; r++) o[r] *= ((const half_t*)p.S)[scale_index_single(col + r)];
        }
        if (row < p.M) *(h4*)((half_t*)p.C + (size_t)row * p.N + col) = o;
      } else {
        const int strip = strip0 + b / MB;
        if (strip >= n_strips) continue;
        // Register r of lane (row, kg) holds slot 4 kg + r, column 16j + 8h + 2s + e
        // of the strip's block, e = kg / 2, j = 2 (kg % 2) + r / 2, h = r % 2.  The
        // lanes of both e, 32 apart, exchange halves and store two columns at a time.
        const int col = 64 * (strip >> 2) + 2 * (strip & 3) + 32 * (kg & 1);
        const int e = kg >> 1;
        unsigned o[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          half_t x = (half_t)v[r];
          if constexpr (!GROUP) x *= ((const half_t*)p.S)[scale_index_single(col + e + 16 * (r >> 1) + 8 * (r & 1))];
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
}

namespace {

// calls f(kernel, LDS bytes) for a set of strips and rows that exists
template <class F>
bool with_rows_kernel(int strips, int blocks, bool group, F f) {
#define ROWS(CS, MB, DEPTH, GROUP)                                               \
  if (strips == CS && blocks == MB && group == GROUP) {                         \
    f(rows_kernel<CS, MB, GROUP, DEPTH>, RowsShape<CS, MB, DEPTH>::kLds);       \
    return true;                                                                \
  }
#define ROWS_OF_BOTH(CS, MB, DEPTH) ROWS(CS, MB, DEPTH, true) ROWS(CS, MB, DEPTH, false)
  ROWS_OF_BOTH(1, 1, 2)
  ROWS_OF_BOTH(2, 1, 2)
  ROWS_OF_BOTH(3, 1, 2)
  ROWS_OF_BOTH(2, 2, 2)
  ROWS_OF_BOTH(3, 2, 1)
  ROWS_OF_BOTH(4, 2, 1)
  ROWS_OF_BOTH(6, 2, 1)
  ROWS_OF_BOTH(2, 3, 1)
  ROWS_OF_BOTH(3, 3, 1)
  ROWS_OF_BOTH(4, 3, 1)
  ROWS_OF_BOTH(5, 3, 1)
  ROWS_OF_BOTH(6, 3, 1)
  ROWS(4, 4, 1, true)  // (never the cheapest with one scale per column)
  ROWS_OF_BOTH(5, 4, 1)
  ROWS_OF_BOTH(6, 4, 1)
  ROWS_OF_BOTH(8, 2, 1)
  ROWS_OF_BOTH(8, 3, 1)
  ROWS_OF_BOTH(8, 4, 1)
#undef ROWS_OF_BOTH
#undef ROWS
  return false;
}

}  // namespace

bool rows_exist(int strips, int blocks, bool group) {
  return with_rows_kernel(strips, blocks, group, [](auto, int) {});
}

int configure_rows_kernels() {
  bool ok = true;
  for (int strips = 1; strips <= kRowsMaxStrips; strips++)
    for (int blocks = 1; blocks <= kRowsMaxBlocks; blocks++)
      for (const bool group : {false, true})
        with_rows_kernel(strips, blocks, group, [&](auto kernel, int lds) {
          ok = ok && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         lds) == hipSuccess;
        });
  return ok ? 0 : 3;
}

int launch_rows(const GemmArgs& a, bool group, int strips, int blocks, hipStream_t stream) {
  GemmArgs b = a;
  b.row_parts = ceil_div(a.M, 16 * blocks);
  b.gpb = ceil_div(a.N / 16, strips) * b.row_parts;
  if (strips == 8 && a.N % 128 != 0) return 2;  // (whole blocks of 64 columns only)
  const bool found = with_rows_kernel(strips, blocks, group, [&](auto kernel, int lds) {
    hipLaunchKernelGGL(kernel, dim3(b.gpb), dim3(64 * kRowsWaves), lds, stream, b);
  });
  return found ? launch_status() : 2;
}

}  // namespace w4a16
