// Dense fp16 GEMM on tiles of many sizes, 32 x 32 to 128 x 256, of which the one is
// taken that fills the compute units best: the problems that are less than a wave
// or two of the tiles of f16_streamk.hip.  Same operands, slabs and order of MFMA
// operands as the kernels there.
//
// Sizes between 64 x 128 and 128 x 256 are there for problems whose 128 x 256 tiles
// leave a quarter to a half of the chip idle (us, operands from memory): 1514 x 3072 x
// 8576, 144 of those 119.9, 256 of 96 x 192 90.8; 701 x 5632 x 832 132 of them 15.7, 240
// of 96 x 192 12.3; 885 x 6912 x 1600 189 of them 27.3, 252 of 128 x 192 23.5.
//
// What bounds a problem of few small tiles is latency: the launch, the first loads, and per
// stage a barrier, the trip of its operands from LDS and, deeper than the ring, that
// from memory: 0.10 us with 32 x 32 tiles, 0.21 with 64 x 64, 0.30 with 64 x 128, 0.04
// to 0.10 more with the chip full (kDnFits).  In slices of 128 x 128 tiles it also paid
// for the slices' meeting, some 4 us of a launch of 9.  Small tiles fill the compute
// units without slices, unless k is deep and C so small that even these leave most of
// the chip idle.  Measured, slices of 128 x 128 tiles against this kernel, operands from
// memory (from the last-level cache), us: 291 x 1280 x 896 9.6 and 4.6 (9.0 and 4.2),
// 1024^3 11.7 and 6.4 (10.3 and 5.4), 777 x 2048 x 1024 12.4 and 9.7 (10.9 and 7.5), 64 x
// 2048 x 4096 14.7 and 10.2 (12.8 and 7.7), 100 x 512 x 10240 29.4 and 11.2 (22.2 and 8.6).
//
// A wave computes half the rows x a quarter (32 x 64 and less: half) of the columns.
// Per 64-deep stage it reads
// all operands of the next stage from LDS while the MFMAs of this one run, so a
// slab is free again as soon as every wave has its operands, and one barrier per
// stage does.  The rings of 32 x 32 to 64 x 64 hold as many slabs as leave room for a
// second workgroup on the compute unit (64 to 72 KiB); from 64 x 128 on a workgroup
// has the unit to itself, and three to six slabs of 24 to 48 KiB (64 x 128: six, 72 KiB
// more in flight than the three that would leave room for a second workgroup: 777 x
// 2048 x 1024 7.9 us, with three 8.2).  Operands loaded straight from memory into
// registers, with the waves along k and no barrier at all, took two to three times as
// long: sixteen rows of 64 bytes per load instruction.
#include <hip/hip_runtime.h>

#include "f16_dense.hpp"
#include "scratch_pool.hpp"

namespace w4a16 {

namespace {

// TM x TN tiles, WM x WN waves
template <int TM, int TN, int WM, int WN, int RING>
struct DnTiles {
  static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
  static constexpr int kRB = TM / 16 / WM, kNJ = TN / 16 / WN;  // operands of a wave per k step
  static constexpr int kOps = 2 * (kRB + kNJ);                  // ... per stage
  static constexpr int kTA = (TM / 8 + kWaves - 1) / kWaves, kTB = TN / 8 / kWaves;  // load instructions per wave and slab
  static constexpr int kSlabA = kTA * kWaves * 1024, kSlab = kSlabA + TN * 128;  // (A: rows past TM stay empty)
  static constexpr int kLoads = kTA + kTB;
  static constexpr int kPitch = TN * 2 + 16;  // bytes per row of the fp16 tile in LDS
  static constexpr int kRingBytes = RING * kSlab, kTileBytes = TM * kPitch;
  static constexpr int kLds = kRingBytes > kTileBytes ? kRingBytes : kTileBytes;
  static constexpr int kPartBytes = TM * TN * 4;
  static_assert(kTB * 8 * kWaves == TN && TM % (16 * WM) == 0 && TN % (16 * WN) == 0, "whole blocks");
  static_assert(kLds <= 160 * 1024 - 256, "LDS of a compute unit");
};

// wait for every LDS read in flight; the registers are named so that they count
// as in use up to here
template <int N>
__device__ __forceinline__ void dn_landed(i4 (&v)[N]) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
#pragma unroll
  for (int i = 4; i < N; i++) asm volatile("" : "+v"(v[i]));
#endif
}
// operands of COUNT neighbouring row blocks of 16
template <int COUNT>
__device__ __forceinline__ void dn_read_blocks(unsigned at, i4* v) {
  if constexpr (COUNT > 0) {
    dn_read_blocks<COUNT - 1>(at, v);
    read_lds16<2048 * (COUNT - 1)>(at, v[COUNT - 1]);
  }
}

}  // namespace

// p.tiles_m x p.tiles_n tiles, all of them in p.ksplit slices (CUT) or whole
template <int TM, int TN, int WM, int WN, int RING, bool CUT>
__global__ __launch_bounds__(64 * WM * WN) void dense_tile_kernel(DenseArgs p) {
  using Sh = DnTiles<TM, TN, WM, WN, RING>;
  constexpr int RB = Sh::kRB, NJ = Sh::kNJ, TA = Sh::kTA, TB = Sh::kTB;
  extern __shared__ __attribute__((aligned(16))) char smem[];  // Sh::kLds
  __shared__ int s_shares;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int kg = lane >> 4;
  const int nu = lane & 15;
  const int wm = wave / WN;
  const int wn = wave % WN;

  int tile, ks = 0;
  if constexpr (CUT)
    dn_slice_coord((int)blockIdx.x, p.tiles_m * p.tiles_n, p.ksplit, &tile, &ks);
  else
    tile = xcd_work_index((int)blockIdx.x, p.tiles_m * p.tiles_n);
  int tm, tn;
  dn_tile_coord(tile, p.tiles_m, p.tiles_n, &tm, &tn);
  const int m0 = TM * tm, n0 = TN * tn;
  const int rows = min(TM, p.M - m0);
  const int cols = min(TN, p.N - n0);  // (192 columns: the last tile may have fewer)
  const __amdgpu_buffer_rsrc_t rA =
      make_rsrc((const char*)p.A + (size_t)m0 * p.K * 2, (unsigned)rows * (unsigned)p.K * 2u);
  const __amdgpu_buffer_rsrc_t rB =
      make_rsrc((const char*)p.B + (size_t)n0 * p.K * 2, (unsigned)cols * (unsigned)p.K * 2u);

  // a wave fetches its share of the rows of A and of B, eight rows per
  // instruction; rows past the end of A repeat the last one (never stored)
  int a_src[TA], b_src[TB];
  {
    const int r8 = lane >> 3, c = (lane & 7) ^ r8;
#pragma unroll
    for (int t = 0; t < TA; t++) {
      const int r = 8 * (TA * wave + t) + r8;
      a_src[t] = r >= TM ? kOob : (r < rows ? r : rows - 1) * p.K * 2 + 16 * c;
    }
#pragma unroll
    for (int t = 0; t < TB; t++) b_src[t] = (8 * (TB * wave + t) + r8) * p.K * 2 + 16 * c;
  }
  // this workgroup's stages (at most 4 slices of at most 2^24 stages: 32 bits do)
  const int all = p.K / kDnStageK;
  const int st0 = CUT ? (int)((unsigned)ks * (unsigned)all / (unsigned)p.ksplit) : 0;
  const int st1 = CUT ? (int)((unsigned)(ks + 1) * (unsigned)all / (unsigned)p.ksplit) : all;
  const int stages = st1 - st0;

  auto issue_slab = [&](int s, int slot) {
    const int inv = s < stages ? 0 : kOob;  // a stage past the end fetches zeros
    const int at = (st0 + s) * (kDnStageK * 2);
    char* const base = smem + slot * Sh::kSlab;
#pragma unroll
    for (int t = 0; t < TA; t++) load_to_lds16(rA, base + (TA * wave + t) * 1024, a_src[t] | inv, at);
#pragma unroll
    for (int t = 0; t < TB; t++)
      load_to_lds16(rB, base + Sh::kSlabA + (TB * wave + t) * 1024, b_src[t] | inv, at);
  };

  // operands of a stage, per k step B then A; where they sit in slab 0
  unsigned a_rd[2], b_rd[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const unsigned sw = 16 * ((4 * h + kg) ^ (nu & 7));
    a_rd[h] = (unsigned)(size_t)smem + (16 * RB * wm + nu) * 128 + sw;
    b_rd[h] = (unsigned)(size_t)smem + Sh::kSlabA + (16 * NJ * wn + nu) * 128 + sw;
  }
  auto read = [&](i4 (&o)[Sh::kOps], unsigned slab) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      dn_read_blocks<NJ>(b_rd[h] + slab, o + h * (RB + NJ));
      dn_read_blocks<RB>(a_rd[h] + slab, o + h * (RB + NJ) + NJ);
    }
  };

  f4 acc[RB][NJ];
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++) acc[i][j] = (f4){0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](i4 (&o)[Sh::kOps]) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(h8, o[h * (RB + NJ) + j]),
              __builtin_bit_cast(h8, o[h * (RB + NJ) + NJ + i]), acc[i][j], 0, 0, 0);
  };

  // Every slot requested; slab 0 landed (loads complete in order), its operands
  // read.  The reads are written by hand (the compiler would wait for every load
  // in flight before each of them); between the reads into a set of registers and
  // the wait that names them stand the MFMAs of the other set and nothing else.
  i4 even[Sh::kOps], odd[Sh::kOps];
#pragma unroll
  for (int r = 0; r < RING; r++) issue_slab(r, r);
  __builtin_amdgcn_s_waitcnt(vmcnt((RING - 1) * Sh::kLoads));
  __builtin_amdgcn_s_barrier();
  read(even, 0);
  dn_landed(even);
  int slot = 0;
  // Stage s, its operands in `cur`: once my loads of the next slab have landed and
  // everybody's have (the barrier, which every wave reaches with its operands of
  // this slab in registers), read the next stage's operands, request the slab
  // after the ring's last in this one's place, and multiply.
  auto stage = [&](int s, i4 (&cur)[Sh::kOps], i4 (&next)[Sh::kOps]) {
    __builtin_amdgcn_s_waitcnt(vmcnt((RING - 2) * Sh::kLoads));
    __builtin_amdgcn_s_barrier();
    const int slot_next = slot == RING - 1 ? 0 : slot + 1;
    __builtin_amdgcn_sched_barrier(0);
    read(next, slot_next * Sh::kSlab);
    issue_slab(s + RING, slot);
    __builtin_amdgcn_sched_barrier(0);
    multiply(cur);
    __builtin_amdgcn_sched_barrier(0);
    dn_landed(next);
    slot = slot_next;
  };
  int s = 0;
  for (; s + 1 < stages; s += 2) {
    stage(s, even, odd);
    stage(s + 1, odd, even);
  }
  if (s < stages) multiply(even);
  // nothing of the ring may still be on its way when LDS is reused
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  // a lane holds, per (i, j), row 16i + nu and four consecutive columns; the tile
  // leaves through LDS as whole rows, the parts of the waves in `waves`
  char* const out = smem + (16 * RB * wm + nu) * Sh::kPitch + (16 * NJ * wn + 4 * kg) * 2;
  half_t* const C = (half_t*)p.C + (size_t)m0 * p.N + n0;
  auto put = [&](int i, int j, f4 v) { *(h4*)(out + 16 * i * Sh::kPitch + 32 * j) = dense_round(v); };
  auto store = [&](int waves) {
    __syncthreads();
    constexpr int PR = TN / 8;  // 16-byte pieces of a row
#pragma unroll
    for (int at0 = 0; at0 < TM * PR; at0 += Sh::kThreads) {
      const int at = at0 + tid;
      const int m = at / PR, c = at % PR;
      if ((TM * PR % Sh::kThreads != 0 && at >= TM * PR) || m >= rows || (TN == 192 && 8 * c >= cols) ||
          !(waves >> (m / (16 * RB) * WN + c / (2 * NJ)) & 1))
        continue;
      // nobody reads C again in this launch
      __builtin_nontemporal_store(*(const i4*)(smem + m * Sh::kPitch + c * 16),
                                  (i4*)(C + (size_t)m * p.N + c * 8));
    }
  };
  if constexpr (!CUT) {
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++) put(i, j, acc[i][j]);
    store(-1);
  } else {
    // slices: as in dense_small_kernel, the pieces of a tile being its waves' parts
    const __amdgpu_buffer_rsrc_t rP = make_rsrc(p.scratch, 0x7fffffffu);
    int* const word = &p.locks[tile * kDnCounterStride];
    const int at = wave * (RB * NJ * 1024) + lane * 16;
    const auto part = [&](int k2) { return (tile * p.ksplit + k2) * Sh::kPartBytes; };
    const auto write_out = [&](int waves) {
      if (waves >> wave & 1) {
#pragma unroll
        for (int e = 0; e < RB * NJ; e++)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, acc[e / NJ][e % NJ]), rP,
                                                 at + e * 1024, part(ks), 16 /* sc1 */);
      }
      __builtin_amdgcn_s_waitcnt(vmcnt(0));  // my stores have been acknowledged
      __syncthreads();
    };
    const int my_share = finish_pieces(1 << ks, p.ksplit, Sh::kWaves);
    write_out(~my_share);
    if (tid == 0) s_shares = finish_arrive(word, p.ksplit, ks, p.finish_polls);
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_shares) == 0) {
      write_out(my_share);
      if (tid == 0) s_shares = finish_abandon(word, p.ksplit, ks);
      __syncthreads();
    }
    const int waves = __builtin_amdgcn_readfirstlane(finish_pieces(s_shares, p.ksplit, Sh::kWaves));
    if (waves >> wave & 1) {
      f4 v[RB * NJ][kDnMaxSlices];  // all of it requested at once
#pragma unroll
      for (int e = 0; e < RB * NJ; e++)
#pragma unroll
        for (int x = 0; x < kDnMaxSlices; x++)
          v[e][x] = x >= p.ksplit ? (f4){0.f, 0.f, 0.f, 0.f}
                    : x == ks     ? acc[e / NJ][e % NJ]
                                  : __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(
                                                               rP, at + e * 1024, part(x), 16 /* sc1 */));
#pragma unroll
      for (int e = 0; e < RB * NJ; e++) {
        f4 sum = v[e][0];
#pragma unroll
        for (int x = 1; x < kDnMaxSlices; x++) sum += v[e][x];
        put(e / NJ, e % NJ, sum);
      }
    }
    store(waves);
    if (tid == 0) finish_leave(word, p.ksplit);
  }
}

namespace {

// calls f(kernel, LDS bytes, threads) for the tile's kernel
template <class F>
void with_tile_kernel(int rows, int cols, bool cut, F f) {
  const auto one = [&](auto shape, auto whole, auto sliced) {
    using Sh = decltype(shape);
    f(cut ? sliced : whole, Sh::kLds, Sh::kThreads);
  };
#define DN_TILE(TM, TN, WM, WN, RING)                                                       \
  if (rows == TM && cols == TN)                                                             \
  return one(DnTiles<TM, TN, WM, WN, RING>{}, dense_tile_kernel<TM, TN, WM, WN, RING, false>, \
             dense_tile_kernel<TM, TN, WM, WN, RING, true>)
  DN_TILE(32, 32, 2, 2, 8);
  DN_TILE(32, 64, 2, 2, 6);
  DN_TILE(64, 64, 2, 4, 4);
  DN_TILE(64, 128, 2, 4, 6);
  if (cut) return;  // only tiles of at most 64 x 128 are cut
  DN_TILE(96, 128, 2, 4, 4);
  DN_TILE(64, 192, 2, 4, 4);
  DN_TILE(96, 192, 2, 4, 3);
  DN_TILE(128, 192, 2, 4, 3);
  DN_TILE(96, 256, 2, 4, 3);
  DN_TILE(128, 256, 2, 4, 3);
#undef DN_TILE
}

}  // namespace

bool dn_tile_exists(int rows, int cols, bool cut) {
  bool found = false;
  with_tile_kernel(rows, cols, cut, [&](auto, int, int) { found = true; });
  return found;
}

hipError_t configure_dense_tiles() {
  hipError_t e = hipSuccess;
  for (const int rows : {32, 64, 96, 128})
    for (const int cols : {32, 64, 128, 192, 256})
      for (const bool cut : {false, true})
        with_tile_kernel(rows, cols, cut, [&](auto kernel, int lds, int) {
          if (e == hipSuccess)
            e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        });
  return e;
}

void launch_dense_tiles(DenseArgs a, const DnTile& t, hipStream_t stream) {
  a.tiles_m = ceil_div(a.M, t.rows);
  a.tiles_n = ceil_div(a.N, t.cols);
  a.ksplit = t.slices;
  with_tile_kernel(t.rows, t.cols, t.slices > 1, [&](auto kernel, int lds, int threads) {
    hipLaunchKernelGGL(kernel, dim3(a.tiles_m * a.tiles_n * t.slices), dim3(threads), lds, stream, a);
  });
}

namespace {

// Costs in us: a launch, a stage of the longest workgroup (dearer the fuller the chip)
// and, whole, workgroups beyond one per compute unit and their stages; in slices the
// launch holds their meeting.  Fitted to every tile on 2500 problems, m = 1 ... 8192, n =
// 256 ... 16384, k = 64 ... 20480; 5 % rms where a tile is within 1.2 times the best.
// Each time is the geometric mean of that with operands from memory, as a model's
// weights are, and of that with operands in the last-level cache: the small tiles, which
// wait for memory, take 1.2 to 1.5 times as long by the first as by the second, slices of
// 128 x 128 1.1 times.  (Fitted to the cache alone, 44 problems of 900 were given tiles
// that took 2 to 19 % longer from memory than the plan's launch: 576 x 1536 x 4544 23.0
// us in 64 x 64, 19.4 in slices; 240 x 3328 x 4096 21.4 and 18.7.  Fitted mostly to memory,
// tiles were given up that were level there and 20 % faster from the cache: 665 x 1280 x
// 3328 12.3 -> 15.6 us.)
struct DnLine {
  double launch, stage, fill;
};
constexpr struct DnFit {
  int rows, cols;
  DnLine whole;
  double more, more_stage;
  DnLine by2, by4;  // (64 x 128: 1.04 times the fit)
} kDnFits[] = {{32, 32, {2.19, 0.093, 0.032}, 0.72, 0.079, {4.41, 0.096, 0.042}, {4.47, 0.090, 0.058}},
               {32, 64, {2.29, 0.138, 0.043}, 0.84, 0.128, {4.84, 0.160, 0.047}, {5.18, 0.142, 0.099}},
               {64, 64, {2.32, 0.191, 0.056}, 0.77, 0.179, {5.25, 0.204, 0.062}, {5.44, 0.192, 0.125}},
               {64, 128, {3.05, 0.277, 0.088}, 2.18, 0.324, {7.08, 0.295, 0.116}, {7.45, 0.287, 0.206}},
               {96, 128, {3.27, 0.359, 0.093}, 2.04, 0.436, {}, {}},
               {64, 192, {3.17, 0.376, 0.109}, 2.17, 0.451, {}, {}},
               {96, 192, {3.62, 0.471, 0.105}, 2.46, 0.611, {}, {}},
               {128, 192, {4.03, 0.475, 0.196}, 2.92, 0.749, {}, {}},
               {96, 256, {4.04, 0.531, 0.205}, 3.09, 0.828, {}, {}},
               {128, 256, {4.46, 0.594, 0.294}, 4.30, 1.020, {}, {}}};

// workgroups beyond one per compute unit: half way between the rounds they make and
// their share of one
double dn_more(int wgs, int cus) {
  const double r = (double)wgs / cus;
  return r > 1.0 ? 0.5 * (ceil_div(wgs, cus) + r) - 1.0 : 0.0;
}

double dn_cost(const DnFit& f, int tiles, int stages, int slices, int cus) {
  const double r = (double)tiles * slices / cus, fill = r < 1.0 ? r : 1.0;
  const DnLine& l = slices == 1 ? f.whole : slices == 2 ? f.by2 : f.by4;
  const double cost = l.launch + ceil_div(stages, slices) * (l.stage + l.fill * fill);
  const double more = slices == 1 ? dn_more(tiles, cus) : 0.0;
  return cost + more * (f.more + f.more_stage * stages);
}

// ... and of the launch that would compute the problem otherwise (3 % rms)
double dn_plan_cost(const DnLaunch& l, int stages, int cus) {
  const double r = (double)l.tiles * l.slices / cus, fill = r < 1.0 ? r : 1.0;
  const double more = dn_more(l.tiles, cus);
  if (l.cols == 128) {
    const double each = (double)stages / l.slices;
    return l.slices == 1   ? 3.17 + 0.43 * fill + stages * (0.424 + 0.095 * fill)
           : l.slices == 2 ? 7.23 + each * (0.367 + 0.213 * fill)
           : l.slices == 3 ? 8.00 + each * (0.261 + 0.349 * fill)
                           : 7.80 + each * (0.370 + 0.261 * fill);
  }
  if (l.rows == 128)
    return l.waves == 4 ? 5.52 + stages * (0.585 + 0.251 * fill)
                        : 4.06 + 0.46 * fill + stages * (0.588 + 0.270 * fill);
  return l.waves == 4 ? 0.13 + 8.17 * fill + 1.87 * more + stages * (1.186 + 0.248 * fill + 1.92 * more)
                      : 2.59 + 4.68 * fill + 6.99 * more + stages * (1.102 + 0.379 * fill + 1.66 * more);
}

}  // namespace

// The cheapest tile, if it is 1 % cheaper than the plan's slices, 3 % than its whole
// tiles and 7 % than those of 256 x 256.  In 2 or 4 slices (waves share a tile unevenly
// with 3) no more than the plan, at most one workgroup per compute unit.  3000 other
// problems for which this or the line before it (one fit, to operands in the cache)
// takes a tile: operands from memory 1.47 times the speed of the plan's launches, 76
// problems more than 2 % slower, the worst by 13 %; by the line before 1.45 times, 165
// slower, the worst by 32 %.  In the cache 1.59 times and one slower; before 1.57 and 62.
DnTile dn_tile(int m, int n, int k, int cus, const DnLaunch& plan) {
  const int stages = k / kDnStageK;
  DnTile best = {0, 0, 0};
  double limit = dn_plan_cost(plan, stages, cus) / (plan.slices > 1 ? 1.01 : plan.rows == 256 ? 1.07 : 1.03);
  for (const DnFit& f : kDnFits) {
    const int tiles = ceil_div(m, f.rows) * ceil_div(n, f.cols);
    if (tiles > 4 * cus) continue;  // (never the best there)
    for (int s = 1; s <= (f.by2.launch > 0 ? plan.slices : 1); s *= 2) {
      if (s > 1 && (tiles * s > cus || tiles > kMaxCounters / kDnCounterStride)) break;
      if (s > 1 && f.cols == 128 && 4 * tiles * s > 3 * cus) break;  // (0.9 to 1.3 times the fit there)
      const double c = dn_cost(f, tiles, stages, s, cus);
      if (c < limit) {
        best = {f.rows, f.cols, s};
        limit = c;
      }
    }
  }
  return best;
}

}  // namespace w4a16
