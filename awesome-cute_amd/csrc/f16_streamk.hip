// Dense fp16 GEMM with a stream-K tail for gfx950: C (m x n, row-major) =
// A (m x k, row-major) * B^T with B given as n rows of k ("TN": both operands
// k-contiguous), fp32 accumulation, alpha = 1, beta = 0 -- the problem of the
// reference's gemm/streamk_gemm (gemm_streamk.cu:8-110), with the same split
// of the output tiles into a data-parallel part and a stream-K part
// (dp_sk_block.h:82-128, strategy sk1tile_dp): tiles that fill whole waves of
// compute units are computed by one workgroup each; the tiles of the last,
// partial wave are cut along k into slices, one workgroup per slice, and the
// slices of a tile meet through fp32 partial sums in memory and a counter.
// Unlike the reference's turnstile (gemm_streamk.h:562-590: every block waits
// for the one before it) nobody waits for a turn: a slice writes what others
// will add up through to memory and arrives, and the slices of a tile finish it
// together, each a share of it, or leave their share to the last arrival when
// the others do not come within a bounded wait (finish_arrive).
//
// dense_kernel: whole tiles, 256 x 256 or (too few of them for the compute
// units) 128 x 256, unless k is shallow, and 128 x 256 in two slices where k is
// deep.  A workgroup of four waves, one per SIMD, each with a 128 x 128 fp32
// accumulator (all 256 AGPRs): a wave per quarter of the tile, or two waves per
// 128 columns, each taking every other k step, their sums added through LDS at
// the end.  The main loop is one assembly statement per tile shape, written by
// gen_dense.py, which documents the schedule and the registers; the build runs it.
//
// dense_small_kernel: eight waves, two per SIMD, of half the tile's rows and a
// quarter of its columns each.  128 x 128 tiles, whole or in slices: the problems
// with few tiles, and the stream-K tiles of the others, every 256 x 256 tile of the
// partial wave as four of its own.  And the large whole tiles over a shallow k, where
// its shorter start and end count for more than dense_kernel's loop.
//
// Problems that take one launch of these go to f16_tiles.hip where tiles of another
// size are cheaper (dn_tile there).
//
// In both, B is the first MFMA operand and A the second, so
// v_mfma_f32_16x16x32_f16 yields D[n][m]; lane l = 16kg + nu of an operand holds
// k = 8kg ... 8kg+7 of row nu.  Per 64-deep stage the workgroup brings a slab of
// A and of B rows into a ring of LDS slots with buffer loads that write LDS
// directly (16 bytes per lane, lane l at 16*l).  Eight lanes fetch the whole
// 128-byte k run of a row -- one cache line; with 64-byte runs every line came
// in twice and the loads alone bounded the kernel -- so a slab is row-major with
// 128-byte rows.  To keep the operand reads (lane (kg, nu): 16 bytes at chunk
// 4h + kg of row nu, one ds_read_b128) free of bank conflicts, the chunk stored
// at position c of row r is chunk c ^ (r % 8); since the hardware fixes where a
// lane's bytes land, the swizzle is applied to the address the lane fetches.
//
// What bounds it: LDS and the way into it, then the board's power.  The large
// tiles with eight waves of 128 x 64 take twelve operand reads per 32 MFMAs, with
// 128 x 128 per wave 16 per 64: 4096^3 101 -> 96 us, 8192 x 8192 x 2048 217 -> 208,
// where the operands stay in the last-level cache (the matrix pipe is then busy 76 %
// of the cycles and LDS reads 21 %); 8192^3, at the power limit, 1.39 PFLOP/s
// either way.  The small tiles
// wait for operands: a compute unit takes in a stage's 32 KiB at 90 to 120 GB/s
// from L2, 57 where A and B come from memory.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <mutex>
#include <type_traits>

#include "../../include/streamk_amd.h"
#include "f16_dense.hpp"
#include "scratch_pool.hpp"
#include "w4a16_common.hpp"

namespace w4a16 {

namespace {

constexpr int kDnTile = 256;     // rows and columns of the large tile of C

// Tiles of dense_kernel, TM rows and 256 columns: 256 x 256 or 128 x 256
template <int TM>
struct DnShape {
  static constexpr int kWK = 256 / TM;          // waves that share a 128 x 128 part's k steps
  static constexpr int kSlabA = TM * 128;
  static constexpr int kSlab = kSlabA + 256 * 128;
  static constexpr int kRing = kWK == 2 ? 3 : 2;
  static constexpr int kSteps = 2 / kWK;        // k steps of a wave per slab
  static constexpr int kTA = kSlabA / 4096;     // load instructions per wave and slab
  static constexpr int kTB = 256 * 128 / 4096;
  static constexpr int kNF = 8 / kWK;           // row blocks of 16 a wave finishes
  static constexpr int kPitch = 256 * 2 + 16;   // bytes per row of the fp16 tile in LDS
  static constexpr int kRingBytes = kRing * kSlab, kTileBytes = TM * kPitch;
  static constexpr int kLds = kRingBytes > kTileBytes ? kRingBytes : kTileBytes;
  static constexpr int kPartBytes = TM * 256 * 4;
  static_assert(kWK == 1 || kLds >= 128 * 1024, "room for the sums that waves hand each other");
};
// Tiles of dense_small_kernel: 128 x 128, 128 x 256 or 256 x 256
template <int TM, int TN>
struct DnSmall {
  static constexpr int kRB = TM / 32;           // row blocks of 16 of a wave
  static constexpr int kNJ = TN / 64;           // operands of 16 columns of a wave
  static constexpr int kSlabA = TM * 128;
  static constexpr int kSlab = kSlabA + TN * 128;
  // A stage of a small tile is shorter than a load's way from L2 (0.4 us of MFMAs
  // for 128 x 128), so its slabs are requested further ahead.
  static constexpr int kRing = TN == 128 ? 4 : TM == 128 ? 3 : 2;
  static constexpr int kTA = TM / 64;           // load instructions per wave and slab
  static constexpr int kLoads = kTA + kNJ;
  static constexpr int kPitch = TN * 2 + 16;
  static constexpr int kRingBytes = kRing * kSlab, kTileBytes = TM * kPitch;
  static constexpr int kLds = kRingBytes > kTileBytes ? kRingBytes : kTileBytes;
  static constexpr int kPartBytes = TM * TN * 4;
};
constexpr int kDnMaxSlots = 256;  // slices in flight per launch
constexpr int kDnPairK = 7168;    // depth from which 128 x 256 tiles in two slices beat 128 x 128 ones
constexpr int kDnRunsK = 6144;    // depth from which 128 x 256 tiles are not dealt out in runs, see there

// wait until at most PENDING later LDS reads are outstanding; `v` is the
// operand the wait is for
template <int PENDING>
__device__ __forceinline__ void dn_wait(i4& v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v) : "n"(PENDING));
#endif
}
// wait for every LDS read in flight; the operand registers are named so that
// they count as in use up to here
__device__ __forceinline__ void drain_reads(i4 (&a)[2], i4 (&b)[2], i4 (&f)[4]) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(a[0]), "+v"(a[1]), "+v"(b[0]), "+v"(b[1]), "+v"(f[0]), "+v"(f[1]), "+v"(f[2]),
                 "+v"(f[3]));
#endif
}
__device__ __forceinline__ void drain_reads(i4 (&a)[4], i4 (&b)[4], i4 (&f)[4]) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]),
                 "+v"(b[3]), "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]));
#endif
}
// s_waitcnt vmcnt(n) lgkmcnt(0) (gfx9 encoding)
constexpr int dn_vm_lgkm0(int n) { return (n & 15) | (7 << 4) | (0 << 8) | ((n >> 4) << 14); }

}  // namespace

// Pieces of an fp16 tile from LDS to C with 16-byte stores, by THREADS threads:
// what `mine(row, operand of 16 columns)` says.
template <int TM, int TN, int PITCH, int THREADS, class Mine>
__device__ __forceinline__ void dense_store_tile(const char* smem, half_t* C, int N, int rows,
                                                 Mine mine) {
  constexpr int PR = TN / 8;  // 16-byte pieces of a row
#pragma unroll 8
  for (int it = 0; it < TM * PR / THREADS; it++) {
    const int at = it * THREADS + (int)threadIdx.x;
    const int m = at / PR, c16 = at % PR;
    if (m < rows && mine(m, c16 / 2)) {
      const i4 v = *(const i4*)(smem + m * PITCH + c16 * 16);
      // nobody reads C again in this launch: keep it out of the way of A and B in L2
      __builtin_nontemporal_store(v, (i4*)(C + (size_t)m * N + c16 * 8));
    }
  }
}

// A whole tile to C: the waves' row blocks (NF each, `sums(i, o)` rounded to `out`,
// NO operands of 16 columns) through LDS in two halves, so that the second half
// is rounded and written to LDS while the first is on its way to memory.  Rows
// r NF 16 ... of the tile belong to one row of waves.
template <int TM, int TN, int PITCH, int THREADS, int NF, int NO, class Sums>
__device__ __forceinline__ void dense_write_tile(const char* smem, char* out, half_t* C, int N, int rows,
                                                 Sums sums) {
  constexpr int PR = TN / 8;     // 16-byte pieces of a row
  constexpr int RUN = 8 * NF;    // rows of a wave in one half
#pragma unroll
  for (int half = 0; half < 2; half++) {
#pragma unroll
    for (int i = half * NF / 2; i < (half + 1) * NF / 2; i++)
#pragma unroll
      for (int o = 0; o < NO; o++) {
        const f4 v = sums(i, o);
        *(h4*)(out + 16 * i * PITCH + 32 * o) =
            (h4){(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
      }
    __syncthreads();
#pragma unroll 8
    for (int it = 0; it < TM / 2 * PR / THREADS; it++) {
      const int at = it * THREADS + (int)threadIdx.x;
      const int r = at / PR, c16 = at % PR;
      const int m = r / RUN * (2 * RUN) + half * RUN + r % RUN;
      if (m < rows) {
        const i4 v = *(const i4*)(smem + m * PITCH + c16 * 16);
        // nobody reads C again in this launch: keep it out of the way of A and B in L2
        __builtin_nontemporal_store(v, (i4*)(C + (size_t)m * N + c16 * 8));
      }
    }
  }
}

// SLICED (128 rows): every tile is cut into p.ksplit slices of the k range,
// which finish it together.
template <int TM, bool SLICED>
__global__ __launch_bounds__(256) void dense_kernel(DenseArgs p) {
  static_assert(!SLICED || TM == 128, "");
  extern __shared__ __attribute__((aligned(16))) char smem[];  // DnShape<TM>::kLds
  using Shape = DnShape<TM>;
  constexpr int WK = Shape::kWK, NF = Shape::kNF, TA = Shape::kTA, TB = Shape::kTB;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int kg = lane >> 4;
  const int nu = lane & 15;
  const int wm = WK == 1 ? wave >> 1 : 0;  // 128-row half of the tile
  const int wn = wave & 1;                 // 128-column half
  const int wk = WK == 1 ? 0 : wave >> 1;  // which of the k steps

  // every XCD gets a contiguous run of tile numbers (a placement hint only)
  // (neighbouring tiles of one k range, so that they share rows of A and B)
  // ... except 128 x 256 tiles over a deep k that the XCDs cannot share evenly: a
  // run of 16 or 17 tiles that begins anywhere in a row of a panel reads up to
  // eight tiles' rows of B, every eighth tile one or two (1306 x 3072 x 7232 90.2
  // us, so 79.2; 1152 x 4352 x 8192 106.7 and 102.9; at k = 5376 58.4 and 59.1)
  const bool runs = SLICED || TM == 256 || (p.dp_tiles & 7) == 0 || p.K < kDnRunsK;
  const int work = runs ? xcd_work_index((int)blockIdx.x, SLICED ? p.dp_tiles * p.ksplit : p.dp_tiles)
                        : (int)blockIdx.x;
  const int ks = SLICED ? work / p.dp_tiles : 0;
  const int tile = SLICED ? work - ks * p.dp_tiles : work;
  int tm, tn;
  dn_tile_coord(tile, p.tiles_m, p.tiles_n, &tm, &tn);
  const int m0 = tm * TM;
  const int n0 = tn * 256;
  const int rows = min(TM, p.M - m0);

  // this workgroup's slabs [first, last) of the K/64
  const int slabs_all = p.K / kDnStageK;
  const int first = SLICED ? (int)((unsigned)ks * (unsigned)slabs_all / (unsigned)p.ksplit) : 0;
  const int last =
      SLICED ? (int)((unsigned)(ks + 1) * (unsigned)slabs_all / (unsigned)p.ksplit) : slabs_all;
  const int skip = first * (kDnStageK * 2);  // bytes of a row before them
  i4 ra_words = rsrc_words((const char*)p.A + (size_t)m0 * p.K * 2 + skip,
                           (unsigned)rows * (unsigned)p.K * 2u - (unsigned)skip);
  i4 rb_words = rsrc_words((const char*)p.B + (size_t)n0 * p.K * 2 + skip,
                           256u * (unsigned)p.K * 2u - (unsigned)skip);

  // wave w fetches the w-th quarter of the A rows and of the B rows of a slab,
  // eight rows per instruction: lane (r = lane/8, c = lane%8) lands at [r][c] and
  // fetches chunk c ^ r of its row.  Rows past the end of A repeat the last row
  // (never stored).
  int src[TA + TB];
  {
    const int r8 = lane >> 3, c = (lane & 7) ^ r8;
#pragma unroll
    for (int t = 0; t < TA + TB; t++) {
      int r = 8 * (t < TA ? TA * wave + t : TB * wave + t - TA) + r8;
      if (t < TA && r >= rows) r = rows - 1;
      src[t] = r * p.K * 2 + 16 * c;
    }
  }
  const int slabs = last - first;
  int s_at = 0;  // byte offset of the next slab to request

  // LDS: where this wave's loads of slot 0 go, and where its operand reads of
  // every slot and step start
  const int lds = (int)(size_t)smem;
  const int lds_a = lds + wave * TA * 1024, lds_b = lds + Shape::kSlabA + wave * TB * 1024;
  constexpr int kReads = Shape::kRing * Shape::kSteps;
  int a_rd[kReads], b_rd[kReads];
#pragma unroll
  for (int j = 0; j < kReads; j++) {
    const int c = 4 * (WK == 1 ? j % Shape::kSteps : wk) + kg;
    const int at = lds + j / Shape::kSteps * Shape::kSlab + nu * 128 + 16 * (c ^ (nu & 7));
    a_rd[j] = at + 128 * wm * 128;
    b_rd[j] = at + Shape::kSlabA + 128 * wn * 128;
  }

  f4 acc[8][8];
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (WK == 1) {
#include "f16_dense_256x256.inc"
  } else {
#include "f16_dense_128x256.inc"
  }
#else  // the host pass only needs the launch stub
  (void)slabs, (void)s_at, (void)lds_a, (void)lds_b, (void)src;
  (void)a_rd, (void)b_rd, (void)ra_words, (void)rb_words;
  for (auto& r : acc)
    for (auto& v : r) v = (f4){0.f, 0.f, 0.f, 0.f};
#endif
  // (nothing is on its way into LDS or registers any more)
  __syncthreads();

  // A lane holds, per (i, o), row 16i + nu and four consecutive columns.  Two
  // waves that share k steps hand each other the four row blocks they will not
  // finish and add; then the fp16 tile goes through LDS.
  constexpr int kPitch = Shape::kPitch;
  char* const out = smem + (128 * wm + 64 * wk + nu) * kPitch + (128 * wn + 4 * (lane >> 4)) * 2;
  half_t* const C = (half_t*)p.C + (size_t)m0 * p.N + n0;
  if constexpr (WK == 1) {
    dense_write_tile<TM, 256, kPitch, 256, NF, 8>(smem, out, C, p.N, rows,
                                                  [&](int i, int o) { return acc[i][o]; });
  } else {
    f4* const swap = (f4*)smem;
    f4 fin[NF][8];
    const auto add_up = [&](auto KEEP) {
      constexpr int keep = decltype(KEEP)::value;
#pragma unroll
      for (int i = 0; i < NF; i++)
#pragma unroll
        for (int o = 0; o < 8; o++) swap[((wave * NF + i) * 8 + o) * 64 + lane] = acc[NF - keep + i][o];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NF; i++)
#pragma unroll
        for (int o = 0; o < 8; o++)
          fin[i][o] = acc[keep + i][o] + swap[(((wave ^ 2) * NF + i) * 8 + o) * 64 + lane];
    };
    if (wk == 0)
      add_up(std::integral_constant<int, 0>{});
    else
      add_up(std::integral_constant<int, NF>{});
    __syncthreads();
    if constexpr (!SLICED) {
      dense_write_tile<TM, 256, kPitch, 256, NF, 8>(smem, out, C, p.N, rows,
                                                    [&](int i, int o) { return fin[i][o]; });
    } else {
      // as in dense_small_kernel, with eight pieces of half the columns of a row
      // block (operands 4 (e % 2) ... + 3 of block e / 2 of every wave)
      __shared__ int s_shares;
      const __amdgpu_buffer_rsrc_t rP = make_rsrc(p.scratch, 0x7fffffffu);
      int* const word = &p.locks[tile * kDnCounterStride];
      const int at = wave * (NF * 8 * 1024) + lane * 16;
      const auto part = [&](int k2) { return (tile * p.ksplit + k2) * Shape::kPartBytes; };
      const auto write_out = [&](int which) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
          if (!(which >> e & 1)) continue;
#pragma unroll
          for (int o = 4 * (e & 1); o < 4 * (e & 1) + 4; o++)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, fin[e >> 1][o]), rP,
                                                   at + (8 * (e >> 1) + o) * 1024, part(ks), 16 /* sc1 */);
        }
        __builtin_amdgcn_s_waitcnt(vmcnt(0));  // my stores have been acknowledged
        __syncthreads();
      };
      const int my_share = finish_pieces(1 << ks, p.ksplit, 8);
      write_out(0xff & ~my_share);
      if (tid == 0) s_shares = finish_arrive(word, p.ksplit, ks, p.finish_polls);
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(s_shares) == 0) {
        write_out(my_share);
        if (tid == 0) s_shares = finish_abandon(word, p.ksplit, ks);
        __syncthreads();
      }
      const int pieces = __builtin_amdgcn_readfirstlane(finish_pieces(s_shares, p.ksplit, 8));
      // two slices: the other one's sums of half my pieces requested at once
#pragma unroll
      for (int h = 0; h < 2; h++) {
        f4 v[4][4];
#pragma unroll
        for (int e = 4 * h; e < 4 * h + 4; e++) {
          if (!(pieces >> e & 1)) continue;
#pragma unroll
          for (int o = 0; o < 4; o++)
            v[e & 3][o] = __builtin_bit_cast(
                f4, __builtin_amdgcn_raw_buffer_load_b128(
                        rP, at + (8 * (e >> 1) + 4 * (e & 1) + o) * 1024, part(1 - ks), 16 /* sc1 */));
        }
#pragma unroll
        for (int e = 4 * h; e < 4 * h + 4; e++) {
          if (!(pieces >> e & 1)) continue;
#pragma unroll
          for (int o = 0; o < 4; o++)  // (a sum of two does not depend on their order)
            *(h4*)(out + 16 * (e >> 1) * kPitch + 32 * (4 * (e & 1) + o)) =
                dense_round(fin[e >> 1][4 * (e & 1) + o] + v[e & 3][o]);
        }
      }
      __syncthreads();
      // (row 64 (m / 64) + 16 i + ..., operand c % 8 of its wave)
      dense_store_tile<TM, 256, kPitch, 256>(smem, C, p.N, rows, [&](int m, int c) {
        return pieces >> (2 * ((m >> 4) & 3) + ((c >> 2) & 1)) & 1;
      });
      if (tid == 0) finish_leave(word, p.ksplit);
    }
  }
}

// CUT: the tiles are cut into slices, or are quarters of the plan's.  (One
// kernel for both took whole tiles 0.25 us longer, 8.5 -> 8.75 us at 2048 x 2048
// x 512.)
// PAIRED (whole tiles): the sums in the order that dense_kernel adds them up in
// two slices, the even and the odd k steps of either half of the k range by
// themselves, so that a problem which runs in such slices where there is scratch
// for them has the same bits where there is none.
template <int TM, int TN, bool CUT, bool PAIRED>
__global__ __launch_bounds__(512) void dense_small_kernel(DenseArgs p) {
  static_assert(!(CUT && PAIRED) && (TM * TN == 128 * 128 || !(CUT || PAIRED)), "");
  extern __shared__ __attribute__((aligned(16))) char smem[];  // DnSmall<TM, TN>::kLds
  using Sh = DnSmall<TM, TN>;
  constexpr int RB = Sh::kRB, NJ = Sh::kNJ, TA = Sh::kTA;
  __shared__ int s_shares;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int kg = lane >> 4;
  const int nu = lane & 15;
  const int wm = wave >> 2;  // row half of the tile
  const int wn = wave & 3;   // column quarter

  // Every XCD gets a contiguous run of slices or of tile numbers (a placement
  // hint only)
  int tile, ks = 0, ksplit = 1, cut = 0;
  if constexpr (CUT) {
    dn_slice_coord((int)blockIdx.x, p.sk_tiles, p.ksplit, &cut, &ks);
    tile = p.dp_tiles + (p.quarters ? cut >> 2 : cut);
    ksplit = p.ksplit;
  } else {
    tile = xcd_work_index((int)blockIdx.x, p.dp_tiles);
  }
  int tm, tn;
  dn_tile_coord(tile, p.tiles_m, p.tiles_n, &tm, &tn);
  int m0 = TM * tm, n0 = TN * tn;
  if (CUT && p.quarters) {
    m0 = 256 * tm + 128 * ((cut >> 1) & 1);
    n0 = 256 * tn + 128 * (cut & 1);
  }
  const int rows = min(TM, p.M - m0);
  if (CUT && rows <= 0) return;  // a quarter below the last row, all its slices

  const __amdgpu_buffer_rsrc_t rA =
      make_rsrc((const char*)p.A + (size_t)m0 * p.K * 2, (unsigned)rows * (unsigned)p.K * 2u);
  const __amdgpu_buffer_rsrc_t rB =
      make_rsrc((const char*)p.B + (size_t)n0 * p.K * 2, (unsigned)TN * (unsigned)p.K * 2u);

  // wave w fetches the w-th eighth of the A rows and of the B rows of a slab, as
  // dense_kernel does
  int a_src[TA], b_src[NJ];
  {
    const int r8 = lane >> 3, c = (lane & 7) ^ r8;
#pragma unroll
    for (int t = 0; t < TA; t++) {
      const int r = 8 * (TA * wave + t) + r8;
      a_src[t] = (r < rows ? r : rows - 1) * p.K * 2 + 16 * c;
    }
#pragma unroll
    for (int t = 0; t < NJ; t++) b_src[t] = (8 * (NJ * wave + t) + r8) * p.K * 2 + 16 * c;
  }
  // this workgroup's stages [st0, st1) of the K/64 stages
  const int stages_all = p.K / kDnStageK;
  // (at most 4 slices of at most 2^24 stages: 32 bits do)
  const int st0 = (int)((unsigned)ks * (unsigned)stages_all / (unsigned)ksplit);
  const int st1 = (int)((unsigned)(ks + 1) * (unsigned)stages_all / (unsigned)ksplit);
  const int stages = st1 - st0;

  auto issue_slab = [&](int s, int slot) {
    const int inv = s < stages ? 0 : kOob;  // a stage past the end fetches zeros
    const int at = (st0 + s) * (kDnStageK * 2);
    char* base = smem + slot * Sh::kSlab;
#pragma unroll
    for (int t = 0; t < TA; t++) load_to_lds16(rA, base + (TA * wave + t) * 1024, a_src[t] | inv, at);
#pragma unroll
    for (int t = 0; t < NJ; t++)
      load_to_lds16(rB, base + Sh::kSlabA + (NJ * wave + t) * 1024, b_src[t] | inv, at);
  };

  f4 acc[RB][NJ];
  f4 odd[PAIRED ? RB : 1][NJ];  // of the odd k steps
  auto start = [&] {
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        acc[i][j] = (f4){0.f, 0.f, 0.f, 0.f};
        if constexpr (PAIRED) odd[i][j] = (f4){0.f, 0.f, 0.f, 0.f};
      }
  };
  start();

  i4 w[2][NJ]; // B operands of the two k steps of a stage
  i4 af[4];    // ring of A operands, three ahead of the MFMAs
  // operand addresses in slab 0 for the two k steps
  unsigned a_rd[2], b_rd[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const unsigned sw = 16 * ((4 * h + kg) ^ (nu & 7));
    a_rd[h] = (unsigned)(size_t)smem + (16 * RB * wm + nu) * 128 + sw;
    b_rd[h] = (unsigned)(size_t)smem + Sh::kSlabA + (16 * NJ * wn + nu) * 128 + sw;
  }
  auto read_b = [&](unsigned at, i4 (&dst)[NJ]) {
    read_lds16<0>(at, dst[0]);
    read_lds16<2048>(at, dst[1]);
    if constexpr (NJ == 4) {
      read_lds16<2 * 2048>(at, dst[2]);
      read_lds16<3 * 2048>(at, dst[3]);
    }
  };

  // prologue: every slot requested; slab 0 landed (loads complete in order); its
  // first operands read
#pragma unroll
  for (int r = 0; r < Sh::kRing; r++) issue_slab(r, r);
  __builtin_amdgcn_s_waitcnt(vmcnt((Sh::kRing - 1) * Sh::kLoads));
  __builtin_amdgcn_s_barrier();
  read_b(b_rd[0], w[0]);
  read_lds16<0>(a_rd[0], af[0]);
  read_lds16<2048>(a_rd[0], af[1]);
  read_lds16<4096>(a_rd[0], af[2]);

  // One k step (H) of the stage in slab `cur`.  LDS reads in issue order, with
  // Ai the operand of row block i and primes the prefetches for the step after:
  //   step 0:  | B(step 1) x NJ  A3 | A0' | A1' | A2' |
  //   step 1:  | A3 | barrier, B(next stage) x NJ  A0' | A1' | A2' |
  // (with eight row blocks A4 ... A7 follow A3 in the same way).
  // When row block i is used, the reads issued after Ai may still be pending:
  // three A operands, plus the NJ B reads where those were issued in between
  // (the three row blocks from the one that issues them).
  // The barrier of a stage sits where the first read from the next slab is
  // about to be issued: by then every wave has its own part of that slab (it
  // waits for its loads first) and has issued and received all its reads of
  // the current slab, which the request for the stage after next overwrites.
  auto kstep = [&](auto H, unsigned cur, unsigned nxt, int s, int slot) {
    constexpr int h = decltype(H)::value;
    constexpr int ib = h ? RB - 3 : 0;  // row block that issues the B reads
    const unsigned ac = a_rd[h] + cur;                      // this step, this slab
    const unsigned an = h ? a_rd[0] + nxt : a_rd[1] + cur;  // the step after
    const unsigned bn = h ? b_rd[0] + nxt : b_rd[1] + cur;
#pragma unroll
    for (int i = 0; i < RB; i++) {
      if (i == ib) {
        if (h == 1) {
          // my loads of the next slab (the slabs after it may still be on
          // their way) and my reads of this one
          __builtin_amdgcn_s_waitcnt(dn_vm_lgkm0((Sh::kRing - 2) * Sh::kLoads));
          __builtin_amdgcn_s_barrier();
          issue_slab(s + Sh::kRing, slot);
        }
        read_b(bn, w[h ^ 1]);
      }
      // operand of row block i + 3: of this step, or of the step after
      auto read_a = [&](auto I) {
        constexpr int x = decltype(I)::value;
        read_lds16<(x < RB ? x : x - RB) * 2048>(x < RB ? ac : an, af[x & 3]);
      };
      switch (i) {  // i is a constant after unrolling
        case 0: read_a(std::integral_constant<int, 3>{}); break;
        case 1: read_a(std::integral_constant<int, 4>{}); break;
        case 2: read_a(std::integral_constant<int, 5>{}); break;
        case 3: read_a(std::integral_constant<int, 6>{}); break;
        case 4: read_a(std::integral_constant<int, 7>{}); break;
        case 5: read_a(std::integral_constant<int, 8>{}); break;
        case 6: read_a(std::integral_constant<int, 9>{}); break;
        case 7: read_a(std::integral_constant<int, 10>{}); break;
      }
      if (i >= ib && i <= ib + 2)
        dn_wait<3 + NJ>(af[i & 3]);
      else
        dn_wait<3>(af[i & 3]);
      if (i == 0) {
        // the B operands of this step were requested before A0 was
#pragma unroll
        for (int j = 0; j < NJ; j++) asm volatile("" : "+v"(w[h][j]));
      }
      const h8 a = __builtin_bit_cast(h8, af[i & 3]);
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        f4& sum = PAIRED && h == 1 ? odd[PAIRED ? i : 0][j] : acc[i][j];
        sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, w[h][j]), a, sum, 0, 0, 0);
      }
    }
  };

  int s = 0;     // the stage being computed
  int slot = 0;  // its ring slot
  auto run_to = [&](int stop) {
    for (; s < stop; s++) {
      const int slot_next = slot == Sh::kRing - 1 ? 0 : slot + 1;
      const unsigned cur = slot * Sh::kSlab, nxt = slot_next * Sh::kSlab;
      kstep(std::integral_constant<int, 0>{}, cur, nxt, s, slot);
      kstep(std::integral_constant<int, 1>{}, cur, nxt, s, slot);
      slot = slot_next;
    }
    // The last k step has requested the operands of the stage after it (which
    // may not exist); they are still on their way into w and af.  Those registers
    // stay taken until the reads have landed: the compiler, which believes they
    // were written when the reads were issued and may see no further use, would
    // otherwise hand them to the code below at once, and a late arrival would
    // overwrite what that code keeps there.
    drain_reads(w[0], w[1], af);
  };
  if constexpr (PAIRED) {
    f4 first[RB][NJ];
    run_to(stages / 2);
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++) first[i][j] = acc[i][j] + odd[i][j];
    start();
    run_to(stages);
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++) acc[i][j] = first[i][j] + (acc[i][j] + odd[i][j]);
  } else {
    run_to(stages);
  }
  // Nothing of the ring may still be on its way when LDS is reused.
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  // a lane holds, per (i, j), row 16i + nu and four consecutive columns
  char* const out = smem + (16 * RB * wm + nu) * Sh::kPitch + (16 * NJ * wn + 4 * (lane >> 4)) * 2;
  half_t* const C = (half_t*)p.C + (size_t)m0 * p.N + n0;
  if (!CUT || ksplit == 1) {
    dense_write_tile<TM, TN, Sh::kPitch, 512, RB, NJ>(smem, out, C, p.N, rows,
                                                     [&](int i, int j) { return acc[i][j]; });
    return;
  }

  // ---- slices of other workgroups: every slice writes the fp32 sums that
  // others will add up through to memory (whole 1 KiB lines per wave
  // instruction), waits for the acknowledgement and arrives; the slices then
  // finish the tile together, each its share of the tile's eight pieces (one (i,
  // j) of every wave), all slices added in slice order.
  const __amdgpu_buffer_rsrc_t rP = make_rsrc(p.scratch, 0x7fffffffu);
  int* const word = &p.locks[cut * kDnCounterStride];
  const int at = wave * (8 * 1024) + lane * 16;
  const auto write_out = [&](int which) {
#pragma unroll
    for (int e = 0; e < 8; e++)
      if (which >> e & 1)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, acc[e >> 1][e & 1]), rP,
                                               at + e * 1024, (cut * ksplit + ks) * Sh::kPartBytes,
                                               16 /* sc1 */);
    __builtin_amdgcn_s_waitcnt(vmcnt(0));  // my stores have been acknowledged
    __syncthreads();
  };
  const int my_share = finish_pieces(1 << ks, ksplit, 8);
  write_out(0xff & ~my_share);
  if (tid == 0) s_shares = finish_arrive(word, ksplit, ks, p.finish_polls);
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(s_shares) == 0) {
    write_out(my_share);
    if (tid == 0) s_shares = finish_abandon(word, ksplit, ks);
    __syncthreads();
  }
  const int pieces = __builtin_amdgcn_readfirstlane(finish_pieces(s_shares, ksplit, 8));
  f4 v[8][kDnMaxSlices - 1];  // all of my pieces requested at once
#pragma unroll
  for (int e = 0; e < 8; e++)
    if (pieces >> e & 1)
#pragma unroll
      for (int x = 0; x < kDnMaxSlices - 1; x++) {
        const int k2 = x < ks ? x : x + 1;
        if (k2 < ksplit)
          v[e][x] = __builtin_bit_cast(
              f4, __builtin_amdgcn_raw_buffer_load_b128(rP, at + e * 1024,
                                                        (cut * ksplit + k2) * Sh::kPartBytes, 16 /* sc1 */));
      }
#pragma unroll
  for (int e = 0; e < 8; e++) {
    if (!(pieces >> e & 1)) continue;
    const f4 own = acc[e >> 1][e & 1];
    f4 sum = ks == 0 ? own : v[e][0];
#pragma unroll
    for (int k2 = 1; k2 < kDnMaxSlices; k2++)
      if (k2 < ksplit) sum += k2 == ks ? own : k2 < ks ? v[e][k2 % (kDnMaxSlices - 1)] : v[e][k2 - 1];
    *(h4*)(out + 16 * (e >> 1) * Sh::kPitch + 32 * (e & 1)) = dense_round(sum);
  }
  __syncthreads();
  // (row 64 (m / 64) + 16 i + ..., operand 2 (c / 2) + j)
  dense_store_tile<128, 128, Sh::kPitch, 512>(
      smem, C, p.N, rows, [&](int m, int c) { return pieces >> (2 * ((m >> 4) & 3) + (c & 1)) & 1; });
  if (tid == 0) finish_leave(word, ksplit);
}

// C = 0 for an empty k range (a kernel rather than a memset, so that the call
// can be captured into a HIP graph like any other)
__global__ void dense_zero_kernel(half_t* C, size_t count) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) C[i] = (half_t)0.f;
}

}  // namespace w4a16

// ---------------------------------------------------------------------------
// Host side: the tile split, the scratch for partial sums, the C ABI.

namespace {

using namespace w4a16;

constexpr int kDnMaxDevices = 16;

thread_local char g_dn_error[256] = "";
thread_local int t_finish_polls = -1;  // streamk_amd_force_finish_polls
thread_local DnTile t_tile = {0, 0, 0};  // streamk_amd_force_tile

void dn_set_error(hipError_t e, const char* what) {
  snprintf(g_dn_error, sizeof(g_dn_error), "%s: %s", what, hipGetErrorString(e));
}

// Partial sums and tile counters of the stream-K tiles come from the scratch
// pool that the W4A16 path uses too: one buffer per (device, stream), sized by
// the launches that need it.
struct DnDevice {
  int cus = 0;
  bool configured = false;
};
std::mutex g_dn_mu;
DnDevice g_dn[kDnMaxDevices];

struct DnPlan {
  int tile_rows, tile_cols, tiles_m, tiles_n, dp_tiles, sk_tiles, ksplit, grid;
};

// Whole waves of tiles go to one workgroup each; the tiles of the partial last
// wave are cut into as many k slices as there are idle compute units per tile
// (at most four, which is what dense_small_kernel has registers for where it adds
// them up), each at least 256 deep.
DnPlan dn_plan(int m, int n, int k, int cus) {
  DnPlan pl;
  // 256 x 256 tiles, unless they would occupy at most half of the compute
  // units: then 128 x 256 tiles, twice as many, and 128 x 128 if that holds
  // for those as well (one workgroup per smaller tile beats k slices of a
  // larger one: no partial sums go through memory)
  pl.tile_rows = pl.tile_cols = kDnTile;
  if (2LL * ceil_div(m, kDnTile) * (n / kDnTile) <= cus) {
    pl.tile_rows = 128;
    if (2LL * ceil_div(m, 128) * (n / kDnTile) <= cus) pl.tile_cols = 128;
  }
  pl.tiles_m = ceil_div(m, pl.tile_rows);
  pl.tiles_n = n / pl.tile_cols;
  const int tiles = pl.tiles_m * pl.tiles_n;
  const int rem = cus > 0 ? tiles % cus : 0;
  int s = 1;
  if (rem > 0) {
    s = cus / rem;
    if (s > kDnMaxSlices) s = kDnMaxSlices;
    if (s > k / 256) s = k / 256;
    while (s > 1 && rem * s > kDnMaxSlots) --s;
    if (s < 1) s = 1;
  }
  pl.ksplit = s;
  pl.sk_tiles = s > 1 ? rem : 0;
  pl.dp_tiles = tiles - pl.sk_tiles;
  pl.grid = pl.dp_tiles + pl.sk_tiles * s;
  return pl;
}

// Whether whole tiles of 256 columns go to dense_kernel's four waves, which read
// less LDS per MFMA, or to dense_small_kernel's eight, which have half as many
// sums each to clear, to add up (128 rows) and to write (1 to 2 us less per
// launch) and request a slab at once.  Four waves save LDS time and power, so
// they are ahead sooner when most of the compute units have a tile, and the
// requests tell where deep operands come from memory and part of the compute
// units have none.  Four and eight waves, us, operands from memory:
//   256 x 256, 145 tiles (1076 x 7424)  k = 512 15.6 and 14.9, 1536 33.7 and 32.8, 2048 41.0 and 41.4,
//                                       4096 78.1 and 81.3, 5376 120.6 and 114.4, 8192 174.7 and 162.0
//              224 tiles (1900 x 7168)  2048 46.7 and 48.6, 5376 130.4 and 126.4, 8192 191.9 and 188.7
//              256 tiles (4096 x 4096)  512 20.2 and 20.2, 1280 36.7 and 38.0, 8192 203.0 and 201.6 (and
//                                       183.6 and 193.6 where they stay in the last-level cache)
//   128 x 256, 132 tiles (1306 x 3072)  512 11.7 and 9.8, 2048 25.8 and 25.2, 3840 45.5 and 43.6, 4096 44.5 and 45.9
//              256 tiles (1000 x 8192)  512 14.7 and 12.9, 2048 33.1 and 33.2, 3072 45.3 and 46.6
bool dn_four_waves(int tile_rows, int tiles, int k, int cus) {
  const bool most = 4 * tiles >= 3 * cus;
  if (tile_rows != kDnTile) return k >= (most ? 3072 : 4096);
  return k >= (most ? 768 : 2048) && (k < 5120 || tiles >= cus);
}

// Whether 128 x 128 tiles are computed two by two, as slices of 128 x 256 ones.
// Problems of 128 x 128 tiles for more than half of the compute units, one
// workgroup each, wait for operands: a tile of 128 x 256 brings half as many rows
// of A per column, so in two slices along k the same workgroups take in three
// quarters of the bytes and run dense_kernel's loop.  The slices' meeting costs
// some 10 us, which a deep k earns back: 128 x 128 against pairs, 777 x 4352 at k =
// 4096 35.3 and 35.9 us, 6144 50.9 and 47.3, 10240 79.9 and 71.1; 513 x 3584 28.6
// and 30.0, 41.4 and 41.3, 65.9 and 62.2; 2048 x 2048 32.9 and 35.4, 48.1 and 47.5,
// 79.2 and 72.5.  At 6144 they are level but for the first, so the line lies above.
// Under capture, and where scratch cannot be had, the tiles are computed whole, in
// the same order of sums and so to the same bits: such a graph names no scratch,
// and may be replayed on any stream beside others.
bool dn_paired(const DnPlan& pl, int k, int cus) {
  return pl.tile_cols == 128 && pl.sk_tiles == 0 && 2 * pl.dp_tiles > cus && k >= kDnPairK;
}

// The launches of a plan; `scratch`: whether pairs have room for their sums
int dn_launches(const DnPlan& pl, int k, int cus, bool scratch, DnLaunch out[2]) {
  int count = 0;
  if (pl.tile_cols == 128) {
    if (pl.sk_tiles > 0)  // (at most one wave of tiles: all of them)
      out[count++] = {128, 128, 8, pl.sk_tiles, pl.ksplit};
    else if (scratch && dn_paired(pl, k, cus))
      out[count++] = {128, 256, 4, pl.dp_tiles / 2, 2};
    else
      out[count++] = {128, 128, 8, pl.dp_tiles, 1};
    return count;
  }
  // The stream-K tiles of large tiles (256 x 256: 128 x 256 ones are less than one
  // wave, and more than half of one) are computed as 128 x 128 quarters in a
  // launch of their own, in slices while that leaves compute units idle: 16
  // tiles of 256 x 256 in four slices are 64 workgroups, a quarter of the chip
  // for a quarter of a tile's time, their quarters 256 (4096 x 4352 x 4096
  // 142 us with one launch for both, 125 with two; 6230 x 3072 x 1280 67 and 52).
  if (pl.sk_tiles > 0) {
    int slices = cus / (4 * pl.sk_tiles);
    if (slices > pl.ksplit) slices = pl.ksplit;
    out[count++] = {128, 128, 8, 4 * pl.sk_tiles, slices < 1 ? 1 : slices};
  }
  if (pl.dp_tiles > 0)
    out[count++] = {pl.tile_rows, 256, dn_four_waves(pl.tile_rows, pl.dp_tiles, k, cus) ? 4 : 8, pl.dp_tiles, 1};
  return count;
}

// The tiles of f16_tiles.hip that compute the problem in place of dn_launches (rows =
// 0: none).  Only in place of one launch, not of pairs of slices, and only in slices
// where that is in slices, and no more of them: the room acquired for their sums then
// holds these as well, and what a stream must have seen before it can be captured
// does not depend on a choice that is a matter of speed.
DnTile dn_tile_for(const DnPlan& pl, int m, int n, int k, int cus) {
  if (t_tile.rows < 0) return {0, 0, 0};
  if (t_tile.rows > 0) {
    DnTile t = t_tile;
    const int most = pl.tile_cols == 128 && pl.sk_tiles > 0 ? pl.ksplit : 1;
    const int tiles = ceil_div(m, t.rows) * ceil_div(n, t.cols);
    if (t.slices > most || tiles > kMaxCounters / kDnCounterStride || !dn_tile_exists(t.rows, t.cols, true))
      t.slices = 1;
    return t;
  }
  DnLaunch launches[2];
  if (dn_paired(pl, k, cus) || dn_launches(pl, k, cus, true, launches) != 1) return {0, 0, 0};
  return dn_tile(m, n, k, cus, launches[0]);
}

int dn_check(int m, int n, int k) {
  if (m < 0 || n < 0 || k < 0) return STREAMK_ERR_SHAPE;
  if (n % kDnTile != 0 || k % kDnStageK != 0) return STREAMK_ERR_SHAPE;
  return STREAMK_OK;
}

}  // namespace

extern "C" {

int streamk_gemm_tn(const void* A, const void* B, void* C, int m, int n, int k, int dev,
                    void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  int rc = dn_check(m, n, k);
  if (rc != STREAMK_OK || m == 0 || n == 0) return rc;
  if (k == 0) {  // an empty sum
    const size_t count = (size_t)m * n;
    hipLaunchKernelGGL(dense_zero_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0,
                       stream, (half_t*)C, count);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      dn_set_error(e, "kernel launch");
      return STREAMK_ERR_RUNTIME;
    }
    return STREAMK_OK;
  }
  // a tile's rows of A and of B are addressed with 32-bit byte offsets
  if ((long long)kDnTile * k * 2 > 0x7fffffffLL) {
    snprintf(g_dn_error, sizeof(g_dn_error), "k = %d is too deep for 32-bit tile offsets", k);
    return STREAMK_ERR_RUNTIME;
  }
  if (dev < 0 || dev >= kDnMaxDevices) {
    snprintf(g_dn_error, sizeof(g_dn_error), "device index %d out of range", dev);
    return STREAMK_ERR_RUNTIME;
  }
  int prev = -1;
  hipError_t e = hipGetDevice(&prev);
  if (e != hipSuccess) {
    dn_set_error(e, "hipGetDevice");
    return STREAMK_ERR_RUNTIME;
  }
  if (prev != dev && (e = hipSetDevice(dev)) != hipSuccess) {
    dn_set_error(e, "hipSetDevice");
    return STREAMK_ERR_RUNTIME;
  }
  rc = STREAMK_ERR_RUNTIME;
  do {
    int cus = 0;
    {
      std::lock_guard<std::mutex> lk(g_dn_mu);
      DnDevice& d = g_dn[dev];
      if (d.cus == 0) {
        e = hipDeviceGetAttribute(&d.cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) {
          d.cus = 0;
          dn_set_error(e, "hipDeviceGetAttribute");
          break;
        }
      }
      cus = d.cus;
      if (!d.configured) {
        e = hipFuncSetAttribute((const void*)dense_kernel<256, false>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, DnShape<256>::kLds);
        if (e == hipSuccess)
          e = hipFuncSetAttribute((const void*)dense_kernel<128, false>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, DnShape<128>::kLds);
        if (e == hipSuccess)
          e = hipFuncSetAttribute((const void*)dense_kernel<128, true>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, DnShape<128>::kLds);
        if (e == hipSuccess)
          e = hipFuncSetAttribute((const void*)dense_small_kernel<128, 128, false, false>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, DnSmall<128, 128>::kLds);
        if (e == hipSuccess)
          e = hipFuncSetAttribute((const void*)dense_small_kernel<128, 128, true, false>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, DnSmall<128, 128>::kLds);
        if (e == hipSuccess)
          e = hipFuncSetAttribute((const void*)dense_small_kernel<128, 128, false, true>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, DnSmall<128, 128>::kLds);
        if (e == hipSuccess)
          e = hipFuncSetAttribute((const void*)dense_small_kernel<128, 256, false, false>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, DnSmall<128, 256>::kLds);
        if (e == hipSuccess)
          e = hipFuncSetAttribute((const void*)dense_small_kernel<256, 256, false, false>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, DnSmall<256, 256>::kLds);
        if (e == hipSuccess) e = configure_dense_tiles();
        if (e != hipSuccess) {
          dn_set_error(e, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
          break;
        }
        d.configured = true;
      }
    }
    const DnPlan pl = dn_plan(m, n, k, cus);
    // only slices exchange anything
    DnLaunch launches[2];
    int count = dn_launches(pl, k, cus, true, launches);
    const DnTile tile = dn_tile_for(pl, m, n, k, cus);
    ScratchView view = {nullptr, nullptr};
    const DnLaunch& first = launches[0];  // (whole tiles come last)
    if (first.slices > 1) {
      const bool paired = dn_paired(pl, k, cus);
      const size_t bytes = (size_t)first.tiles * first.slices * first.rows * first.cols * 4;
      hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
      const bool may = !paired || (hipStreamIsCapturing(stream, &capture) == hipSuccess &&
                                   capture == hipStreamCaptureStatusNone);
      if (!may || !scratch_acquire(dev, stream, bytes, &view, g_dn_error, sizeof(g_dn_error))) {
        if (!paired) break;
        count = dn_launches(pl, k, cus, false, launches);
      }
    }
    (void)hipGetLastError();  // an earlier call's error is not this launch's
    DenseArgs a;
    a.A = A;
    a.B = B;
    a.C = C;
    a.M = m;
    a.N = n;
    a.K = k;
    a.tiles_m = pl.tiles_m;
    a.tiles_n = pl.tiles_n;
    a.locks = view.counters;
    a.scratch = view.partials;
    a.finish_polls = t_finish_polls < 0 ? kFinishPolls : t_finish_polls;
    if (tile.rows > 0) {
      launch_dense_tiles(a, tile, stream);
      count = 0;  // in place of the plan's launches
    }
    for (int i = 0; i < count; i++) {
      const DnLaunch& l = launches[i];
      const bool pairs = l.cols > pl.tile_cols;
      if (pairs) a.tiles_n = n / l.cols;
      // (tiles in slices, and quarters, are the ones after the whole tiles)
      const bool cut = l.slices > 1 || l.rows < pl.tile_rows;
      a.dp_tiles = pairs ? l.tiles : pl.dp_tiles;
      a.sk_tiles = cut ? l.tiles : 0;
      a.ksplit = l.slices;
      a.quarters = l.rows < pl.tile_rows ? 1 : 0;
      const auto launch = [&](auto kernel, int lds) {
        hipLaunchKernelGGL(kernel, dim3(l.tiles * l.slices), dim3(64 * l.waves), lds, stream, a);
      };
      if (l.waves == 4) {
        if (pairs)
          launch(dense_kernel<128, true>, DnShape<128>::kLds);
        else if (l.rows == 128)
          launch(dense_kernel<128, false>, DnShape<128>::kLds);
        else
          launch(dense_kernel<256, false>, DnShape<256>::kLds);
      } else if (l.cols == 128) {
        if (cut)
          launch(dense_small_kernel<128, 128, true, false>, DnSmall<128, 128>::kLds);
        else if (dn_paired(pl, k, cus))
          launch(dense_small_kernel<128, 128, false, true>, DnSmall<128, 128>::kLds);
        else
          launch(dense_small_kernel<128, 128, false, false>, DnSmall<128, 128>::kLds);
      } else if (l.rows == 128) {
        launch(dense_small_kernel<128, 256, false, false>, DnSmall<128, 256>::kLds);
      } else {
        launch(dense_small_kernel<256, 256, false, false>, DnSmall<256, 256>::kLds);
      }
    }
    e = hipGetLastError();
    if (e != hipSuccess) {
      dn_set_error(e, "kernel launch");
      break;
    }
    rc = STREAMK_OK;
  } while (false);
  if (prev != dev) (void)hipSetDevice(prev);
  return rc;
}

int streamk_amd_check(int m, int n, int k) { return dn_check(m, n, k); }

int streamk_amd_plan(int m, int n, int k, int cus, int* out) {
  const int rc = dn_check(m, n, k);
  if (rc != STREAMK_OK) return rc;
  const DnPlan pl = dn_plan(m, n, k, cus);
  out[0] = pl.tiles_m;
  out[1] = pl.tiles_n;
  out[2] = pl.dp_tiles;
  out[3] = pl.sk_tiles;
  out[4] = pl.ksplit;
  out[5] = pl.grid;
  out[6] = pl.tile_rows;
  out[7] = pl.tile_cols;
  return STREAMK_OK;
}

int streamk_amd_tile(int m, int n, int k, int cus, int* out) {
  out[0] = out[1] = out[2] = 0;
  const int rc = dn_check(m, n, k);
  if (rc != STREAMK_OK || m == 0 || n == 0 || k == 0) return rc;
  const DnTile t = dn_tile_for(dn_plan(m, n, k, cus), m, n, k, cus);
  out[0] = t.rows;
  out[1] = t.cols;
  out[2] = t.slices;
  return STREAMK_OK;
}

int streamk_amd_launches(int m, int n, int k, int cus, int scratch, int* out) {
  if (dn_check(m, n, k) != STREAMK_OK || m == 0 || n == 0 || k == 0) return 0;
  DnLaunch launches[2];
  const int count = dn_launches(dn_plan(m, n, k, cus), k, cus, scratch != 0, launches);
  for (int i = 0; i < count; i++) {
    const DnLaunch& l = launches[i];
    const int fields[5] = {l.rows, l.cols, l.waves, l.tiles, l.slices};
    for (int j = 0; j < 5; j++) out[5 * i + j] = fields[j];
  }
  return count;
}

void streamk_amd_tile_coord(int tile, int tiles_m, int tiles_n, int* out) {
  dn_tile_coord(tile, tiles_m, tiles_n, &out[0], &out[1]);
}

void streamk_amd_slice_coord(int block, int tiles, int slices, int* out) {
  dn_slice_coord(block, tiles, slices, &out[0], &out[1]);
}

void streamk_amd_force_finish_polls(int polls) {
  t_finish_polls = polls < 0 || polls > kFinishPolls ? -1 : polls;
}

void streamk_amd_force_tile(int rows, int cols, int slices) {
  const bool exists = dn_tile_exists(rows, cols, false);
  t_tile = {rows < 0 ? -1 : exists ? rows : 0, exists ? cols : 0,
            slices < 1 ? 1 : slices > kDnMaxSlices ? kDnMaxSlices : slices};
}

long long streamk_amd_release(int dev) { return (long long)scratch_release(dev); }

const char* streamk_amd_last_error(void) { return g_dn_error; }

}  // extern "C"
