// Weight conversion on the GPU: fp16 weights to 4-bit integers, fake weights
// and scales (quantise_*), and fake weights to the packed layout (pack_*), the
// arithmetic of the reference's Layer.pack (marlin.py:92-131) and of its
// tests' quantiser (marlin_test.py:18-40).
//
// Bound: memory.  As a sequence of tensor operations the two took some thirty
// passes over the weight, half of them over 64-bit integers (n = 11008, k =
// 4096: 1712 us for the pair).  Here each is one pass: the quantiser reads a
// weight once (twice where a group does not fit into registers) and writes its
// 6 bytes, the packer reads it once and writes its half byte: 90 us for the pair, 66 of
// it the quantiser, at 5.4 TB/s as is the packer (a copy reaches 5.0 to 5.3).
//
// Every rounding is that of the tensor operations: fp16(w / s) is the rounded
// fp32 quotient rounded once more, the integer is rounded half to even, and
// (q - 8) * s is rounded once.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

#include "../../include/marlin_amd_convert.h"
#include "../../include/marlin_amd_tools.h"
#include "w4a16_common.hpp"

namespace w4a16 {

namespace {

typedef unsigned short us4 __attribute__((ext_vector_type(4)));
typedef unsigned short us8 __attribute__((ext_vector_type(8)));

constexpr int kQThreads = 512;
constexpr int kPThreads = 256;
constexpr int kKeep = 16;  // 8-byte pieces of its group a thread keeps between the two passes

// Bit patterns of non-negative halves order as their values, infinity above
// all numbers and NaN above infinity: an integer maximum hands on a NaN, as
// the tensor operation does.
__device__ __forceinline__ us4 abs_bits(i2 v) {
  return __builtin_bit_cast(us4, v & (i2){0x7fff7fff, 0x7fff7fff});
}
__device__ __forceinline__ us4 max_of(us4 a, us4 b) { return __builtin_elementwise_max(a, b); }
__device__ __forceinline__ us4 shfl_xor_of(us4 v, int mask) {
  i2 x = __builtin_bit_cast(i2, v);
  x[0] = __shfl_xor(x[0], mask);
  x[1] = __shfl_xor(x[1], mask);
  return __builtin_bit_cast(us4, x);
}

__device__ __forceinline__ half_t scale_of(unsigned short max_bits) {
  return (half_t)((float)__builtin_bit_cast(half_t, max_bits) * (float)(2.0 / 15.0));
}

// round(fp16(w / s)) + 8, clamped to 0 ... 15, with r an approximation of
// 1 / s.  The quotient of two halves is either a number of at most 12 bits or
// at least 2^-24 of itself away from one, so a quotient within an fp32 ulp
// that is exact where the true one has 12 bits rounds to the same half; one
// residual step on w * r gives that.  Where the residual is not a number (a
// zero or infinite operand, NaN) the division itself decides.
__device__ __forceinline__ int quantised(half_t w, float s, float r) {
  const float x = (float)w;
  float q = x * r;
  const float e = __builtin_fmaf(-q, s, x);
  q = __builtin_fmaf(e, r, q);
  if (__builtin_expect(!(__builtin_fabsf(e) < __builtin_inff()), 0)) q = x / s;
  const float h = (float)(half_t)q;
  // a NaN becomes 0 and an infinity the largest integer, which wraps (said in so
  // many words: of an integer sum the compiler keeps the clamp at 15)
  const int i = h == __builtin_inff() ? -8 : __float2int_rn(h) + 8;
  return i < 0 ? 0 : i > 15 ? 15 : i;
}

// quantised() of two halves, in bits 0-3 and 16-19.  Numbers are clamped to -8 ...
// 7 as halves and rounded to whole ones by adding 1544: halves from 1024 to 2048 are
// whole, sums are rounded half to even, and the low four bits of 1544 + i are those
// of 8 + i.  Quotients that no half is near (a zero or infinite operand, NaN,
// overflow) go through quantised().
__device__ __forceinline__ int quantised_pair(half_t a, half_t b, float sa, float ra, float sb, float rb) {
  const float x = (float)a, y = (float)b;
  float p = x * ra, q = y * rb;
  p = __builtin_fmaf(__builtin_fmaf(-p, sa, x), ra, p);
  q = __builtin_fmaf(__builtin_fmaf(-q, sb, y), rb, q);
  if (__builtin_expect(!(__builtin_fabsf(p) < 65520.f) || !(__builtin_fabsf(q) < 65520.f), 0))
    return quantised(a, sa, ra) | (quantised(b, sb, rb) << 16);
  const h2 top = {(half_t)7.f, (half_t)7.f}, bottom = {(half_t)-8.f, (half_t)-8.f};
  const h2 whole = {(half_t)1544.f, (half_t)1544.f};
  const h2 v = {(half_t)p, (half_t)q};
  return as_int(__builtin_elementwise_max(__builtin_elementwise_min(v, top), bottom) + whole) & 0x000f000f;
}

template <int N>
struct Columns {  // N columns' scales and their reciprocals
  float s[N], r[N];
  __device__ __forceinline__ void set(int i, half_t v) {
    s[i] = (float)v;
    r[i] = __builtin_amdgcn_rcpf(s[i]);
  }
};

// Four neighbouring elements: fake weights and integers out.  Four and not
// eight, so that the lanes of a store instruction write whole lines of both
// (eight: two instructions that each write every other 16 bytes of the
// integers; n = 11008, k = 4096: 101 us against 70, 5.1 TB/s).
template <class S>
__device__ __forceinline__ void write4(i2 v, const S& c, half_t* fake, int* q) {
  const h4 w = __builtin_bit_cast(h4, v);
  h4 f;
  i4 o;
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const int x = quantised_pair(w[i], w[i + 1], c.s[i], c.r[i], c.s[i + 1], c.r[i + 1]);
    // (1024 + x - 1032 is exact, and the product rounded once)
    const h2 whole = as_h2(x | 0x64006400) - (h2){(half_t)1032.f, (half_t)1032.f};
    const h2 y = whole * (h2){(half_t)c.s[i], (half_t)c.s[i + 1]};
    f[i] = y[0];
    f[i + 1] = y[1];
    o[i] = x & 0xffff;
    o[i + 1] = x >> 16;
  }
  *(h4*)fake = f;
  // (nothing reads the integers soon; the packer reads the fake weights)
  __builtin_nontemporal_store(o, (i4*)q);
}

// (k, n), columns contiguous.  A workgroup takes one group of 4 CL columns, a
// thread four of them and every (512 / CL)-th row.  CL = 64 for groups of up
// to 128 rows, which then stay in registers; CL = 16 for longer ones that are not
// quantised in chunks (in_chunks).
template <int CL>
__global__ __launch_bounds__(kQThreads) void quantise_rows(const half_t* w, int n, int gs,
                                                           half_t* fake, int* q, half_t* s) {
  constexpr int RL = kQThreads / CL;
  constexpr bool KEEP = CL == 64;
  __shared__ us4 part[kQThreads / kWave][CL];
  const int cl = threadIdx.x % CL, rl = threadIdx.x / CL;
  const int c0 = ((int)blockIdx.x * CL + cl) * 4;
  const bool on = c0 < n;
  const size_t base = (size_t)blockIdx.y * gs * n + c0;
  i2 keep[KEEP ? kKeep : 1];
  us4 top = (us4)0;
  if (KEEP) {
#pragma unroll
    for (int i = 0; i < kKeep; i++) {
      const int row = rl + i * RL;
      keep[i] = on && row < gs ? *(const i2*)(w + base + (size_t)row * n) : (i2)0;
    }
#pragma unroll
    for (int i = 0; i < kKeep; i++) top = max_of(top, abs_bits(keep[i]));
  } else if (on) {
#pragma unroll 8
    for (int row = rl; row < gs; row += RL)
      top = max_of(top, abs_bits(*(const i2*)(w + base + (size_t)row * n)));
  }
#pragma unroll
  for (int m = CL; m < kWave; m *= 2) top = max_of(top, shfl_xor_of(top, m));
  if ((threadIdx.x & 63) < CL) part[threadIdx.x / kWave][cl] = top;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kQThreads / kWave; i++) top = max_of(top, part[i][cl]);
  if (!on) return;
  Columns<4> col;
  h4 sv;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    sv[i] = scale_of(top[i]);
    col.set(i, sv[i]);
  }
  if (rl == 0) *(h4*)(s + (size_t)blockIdx.y * n + c0) = sv;
  if (KEEP) {
#pragma unroll
    for (int i = 0; i < kKeep; i++) {
      const int row = rl + i * RL;
      const size_t at = base + (size_t)row * n;
      if (row < gs) write4(keep[i], col, fake + at, q + at);
    }
  } else {
#pragma unroll 4
    for (int row = rl; row < gs; row += RL) {
      const size_t at = base + (size_t)row * n;
      write4(*(const i2*)(w + at), col, fake + at, q + at);
    }
  }
}

// Long groups, (k, n) with columns contiguous, in three launches, so that chunks of
// 128 rows are workgroups of their own: the largest magnitudes of every chunk, the
// scales from them, and the chunks quantised.  The magnitudes lie at the head of q,
// which the last launch overwrites.
constexpr int kChunkRows = 128;

__global__ __launch_bounds__(kQThreads) void chunk_maxima(const half_t* w, int n, int gs, int per_group,
                                                          unsigned short* part) {
  __shared__ us4 top_of[kQThreads / kWave][kWave];
  const int cl = threadIdx.x % kWave, rl = threadIdx.x / kWave;
  const int c0 = ((int)blockIdx.x * kWave + cl) * 4;
  const int g = (int)blockIdx.y / per_group, r0 = ((int)blockIdx.y - g * per_group) * kChunkRows;
  const int rows = gs - r0 < kChunkRows ? gs - r0 : kChunkRows;
  us4 top = (us4)0;
  if (c0 < n) {
    const half_t* const at = w + ((size_t)g * gs + r0) * n + c0;
    i2 v[kKeep];
#pragma unroll
    for (int i = 0; i < kKeep; i++) {
      const int row = rl + i * (kQThreads / kWave);
      v[i] = row < rows ? *(const i2*)(at + (size_t)row * n) : (i2)0;
    }
#pragma unroll
    for (int i = 0; i < kKeep; i++) top = max_of(top, abs_bits(v[i]));
  }
  top_of[rl][cl] = top;
  __syncthreads();
  if (rl != 0 || c0 >= n) return;
#pragma unroll
  for (int i = 1; i < kQThreads / kWave; i++) top = max_of(top, top_of[i][cl]);
  *(us4*)(part + (size_t)blockIdx.y * n + c0) = top;
}

__global__ __launch_bounds__(kQThreads) void chunk_scales(const unsigned short* part, int n, int per_group,
                                                          half_t* s) {
  __shared__ us4 top_of[kQThreads / 16][16];
  const int cl = threadIdx.x % 16, rl = threadIdx.x / 16;
  const int c0 = ((int)blockIdx.x * 16 + cl) * 4;
  us4 top = (us4)0;
  if (c0 < n)
    for (int i = rl; i < per_group; i += kQThreads / 16)
      top = max_of(top, *(const us4*)(part + ((size_t)blockIdx.y * per_group + i) * n + c0));
  top_of[rl][cl] = top;
  __syncthreads();
  if (rl != 0 || c0 >= n) return;
#pragma unroll 8
  for (int i = 1; i < kQThreads / 16; i++) top = max_of(top, top_of[i][cl]);
  h4 sv;
#pragma unroll
  for (int i = 0; i < 4; i++) sv[i] = scale_of(top[i]);
  *(h4*)(s + (size_t)blockIdx.y * n + c0) = sv;
}

__global__ __launch_bounds__(kQThreads) void quantise_chunks(const half_t* w, int n, int gs, int per_group,
                                                             half_t* fake, int* q, const half_t* s) {
  const int c0 = ((int)blockIdx.x * kWave + (int)(threadIdx.x % kWave)) * 4;
  if (c0 >= n) return;
  const int g = (int)blockIdx.y / per_group, r0 = ((int)blockIdx.y - g * per_group) * kChunkRows;
  const int rows = gs - r0 < kChunkRows ? gs - r0 : kChunkRows;
  const size_t base = ((size_t)g * gs + r0) * n + c0;
  const int rl = threadIdx.x / kWave;
  i2 v[kKeep];
#pragma unroll
  for (int i = 0; i < kKeep; i++) {
    const int row = rl + i * (kQThreads / kWave);
    v[i] = row < rows ? *(const i2*)(w + base + (size_t)row * n) : (i2)0;
  }
  const h4 sv = *(const h4*)(s + (size_t)g * n + c0);
  Columns<4> col;
#pragma unroll
  for (int i = 0; i < 4; i++) col.set(i, sv[i]);
#pragma unroll
  for (int i = 0; i < kKeep; i++) {
    const int row = rl + i * (kQThreads / kWave);
    const size_t at = base + (size_t)row * n;
    if (row < rows) write4(v[i], col, fake + at, q + at);
  }
}

struct OneColumn {
  struct Same {
    float v;
    __device__ __forceinline__ float operator[](int) const { return v; }
  } s, r;
};

// The same values stored column by column, (n, k).  T neighbouring threads
// take one group of one column, 4 T k-values at a time: 32 for groups of up to
// 128, the whole workgroup for longer ones.
template <int T>
__global__ __launch_bounds__(kPThreads) void quantise_columns(const half_t* w, int n, int k, int gs,
                                                              half_t* fake, int* q, half_t* s) {
  __shared__ unsigned part[kPThreads / kWave];
  const int groups = k / gs;
  const long long team = (long long)blockIdx.x * (kPThreads / T) + threadIdx.x / T;
  if (T < kPThreads && team >= (long long)n * groups) return;  // whole teams, no barrier below
  const int at0 = (int)(threadIdx.x % T) * 4;
  const size_t base = (size_t)(team / groups) * k + (size_t)(team % groups) * gs;
  const i2 first = at0 < gs ? *(const i2*)(w + base + at0) : (i2)0;
  us4 top = abs_bits(first);
  for (int at = at0 + 4 * T; at < gs; at += 4 * T)
    top = max_of(top, abs_bits(*(const i2*)(w + base + at)));
  unsigned m = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) m = top[i] > m ? top[i] : m;
#pragma unroll
  for (int x = 1; x < (T < kWave ? T : kWave); x *= 2) {
    const unsigned o = __shfl_xor(m, x);
    m = o > m ? o : m;
  }
  if (T > kWave) {
    if ((threadIdx.x & 63) == 0) part[threadIdx.x / kWave] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPThreads / kWave; i++) m = part[i] > m ? part[i] : m;
  }
  const half_t sv = scale_of((unsigned short)m);
  const float sf = (float)sv;
  const OneColumn col = {{sf}, {__builtin_amdgcn_rcpf(sf)}};
  if (at0 == 0) s[(size_t)(team % groups) * n + team / groups] = sv;
  if (at0 < gs) write4(first, col, fake + base + at0, q + base + at0);
  for (int at = at0 + 4 * T; at < gs; at += 4 * T)
    write4(*(const i2*)(w + base + at), col, fake + base + at, q + base + at);
}

// position of column c's scale in the packed order: an 8 x 8 transpose in
// blocks of 64 columns with group scales, {2i, 2i+1} of every 8 gathered in
// blocks of 32 with one scale per column (reference marlin.py:49-55)
__device__ __forceinline__ int scale_slot(int c, bool grouped) {
  if (grouped) return (c & ~63) + 8 * (c & 7) + ((c >> 3) & 7);
  return (c & ~31) + 8 * ((c >> 1) & 3) + 2 * ((c >> 3) & 3) + (c & 1);
}

struct PackArgs {
  const void* w;
  const half_t* scales;
  long long s_group, s_col;
  int* B;
  half_t* s_packed;
  int k, n, gs;  // gs: k-values per scale
  bool grouped;
};

// (k, n), columns contiguous; whole numbers (INTS) or fake weights.  Word
// (t, c, j) of a 16 x 64 block holds rows 2t, 2t+1, 2t+8, 2t+9 of columns
// 16j + c and 16j + c + 8 (reference marlin.py:29-48): thread (t, 8 columns)
// reads those four rows, has one half of eight words, and exchanges four
// halves with the thread of the other eight columns.  Four t and sixteen
// column threads in a wave: a row is read in runs of 256 bytes.  A thread then
// has four c of one j, and exchanges them with the threads of the other three j
// for four j of one c, 16 bytes of B: 32 threads store 512 bytes in a row.
// (Stored as words, every 16 bytes, and quantised one by one: n = 11008, k = 4096,
// weights from memory, 31.2 us; so 23.4, 4.8 TB/s.)
template <bool INTS>
__global__ __launch_bounds__(kPThreads) void pack_rows(PackArgs p) {
  const int t = threadIdx.x & 3;
  const int c0 = ((int)blockIdx.x * (kPThreads / 4) + (int)(threadIdx.x >> 2)) * 8;
  if (c0 >= p.n) return;  // (all threads of an exchange or none: n is a multiple of 64)
  const int kt = blockIdx.y;
  int half[8];
  if constexpr (INTS) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = 16 * kt + 2 * t + (r & 1) + 8 * (r >> 1);
      const int shift = 16 * (r & 1) + 4 * (r >> 1);
      const int* const q = (const int*)p.w + (size_t)row * p.n + c0;
      int v[8];
      *(i4*)v = *(const i4*)q;
      *(i4*)(v + 4) = *(const i4*)(q + 4);
#pragma unroll
      for (int i = 0; i < 8; i++) half[i] = r == 0 ? v[i] : half[i] | (v[i] << shift);
    }
  } else {
    h8 w[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = 16 * kt + 2 * t + (r & 1) + 8 * (r >> 1);
      w[r] = *(const h8*)((const half_t*)p.w + (size_t)row * p.n + c0);
    }
    const int g = 16 * kt / p.gs;
    Columns<8> col;
    half_t sv[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      sv[i] = p.scales[g * p.s_group + (c0 + i) * p.s_col];
      col.set(i, sv[i]);
    }
    if (t == 0 && 16 * kt == g * p.gs) {
      half_t* out = p.s_packed + (size_t)g * p.n;
#pragma unroll
      for (int i = 0; i < 8; i++) out[scale_slot(c0 + i, p.grouped)] = sv[i];
    }
#pragma unroll
    for (int i = 0; i < 8; i++)
      half[i] = quantised_pair(w[0][i], w[1][i], col.s[i], col.r[i], col.s[i], col.r[i]) |
                (quantised_pair(w[2][i], w[3][i], col.s[i], col.r[i], col.s[i], col.r[i]) << 4);
  }
  const int odd = (c0 >> 3) & 1;  // columns 8 ... 15 of their sixteen
  const int j0 = (c0 >> 4) & 1, j1 = (c0 >> 5) & 1;
  int word[4];  // c = i + 4 odd, my j
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int got = __shfl_xor(odd ? half[i] : half[i + 4], 4);
    // even: c = i with the partner's columns above; odd: c = i + 4
    word[i] = odd ? got | (half[i + 4] << 8) : half[i] | (got << 8);
  }
  int pair[2][2];  // c = 2i + j0 + 4 odd; j = its second index + 2 j1
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int got = __shfl_xor(j0 ? word[2 * i] : word[2 * i + 1], 8);
    pair[i][0] = j0 ? got : word[2 * i];
    pair[i][1] = j0 ? word[2 * i + 1] : got;
  }
  i4 out;  // c = 2 j1 + j0 + 4 odd, all j
#pragma unroll
  for (int x = 0; x < 2; x++) {
    const int got = __shfl_xor(j1 ? pair[0][x] : pair[1][x], 16);
    out[x] = j1 ? got : pair[0][x];
    out[2 + x] = j1 ? pair[1][x] : got;
  }
  *(i4*)(p.B + (size_t)kt * 2 * p.n + (c0 >> 6) * 128 + 16 * (2 * j1 + j0 + 4 * odd) + 4 * t) = out;
}

// Fake weights stored column by column, (n, k): a wave takes 64 k-values of a
// 64-column block, eight lanes a column's 128 bytes at a time, and writes four
// rows of B of it completely.  A thread then has eight k-values (low or high
// ones of a row of B, by its lane's lowest bit) of columns 8 i + lane / 8, both
// halves of sixteen columns, and exchanges with its neighbour: the even one takes
// t = 0, 1, the odd one 2, 3, all j of them, 32 bytes in a row.  (With a column per
// lane, whose load instructions touch 64 lines each, n = 11008, k = 4096 took 50
// us, so 27.3.)
__global__ __launch_bounds__(kPThreads) void pack_columns(PackArgs p) {
  const int lane = threadIdx.x & 63;
  const int blk = (int)blockIdx.x;
  const int k0 = ((int)blockIdx.y * (kPThreads / kWave) + (int)(threadIdx.x >> 6)) * 64;
  if (k0 >= p.k) return;
  const int c = blk * 64 + (lane >> 3), chunk = lane & 7, odd = lane & 1;
  const h8* src = (const h8*)((const half_t*)p.w + (size_t)c * p.k + k0) + chunk;
  h8 w[8];
#pragma unroll
  for (int i = 0; i < 8; i++) w[i] = src[(size_t)i * p.k];
  const int g = k0 / p.gs;
  half_t sv[8];
#pragma unroll
  for (int i = 0; i < 8; i++) sv[i] = p.scales[g * p.s_group + (c + 8 * i) * p.s_col];
  if (chunk == 0 && k0 == g * p.gs) {
    half_t* const out = p.s_packed + (size_t)g * p.n;
#pragma unroll
    for (int i = 0; i < 8; i++) out[scale_slot(c + 8 * i, p.grouped)] = sv[i];
  }
  int half[4][4];  // [t][j]: my four bits of both columns
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float s = (float)sv[i], rs = __builtin_amdgcn_rcpf(s);
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int v = quantised_pair(w[i][2 * t], w[i][2 * t + 1], s, rs, s, rs);
      half[t][i >> 1] = (i & 1) == 0 ? v : half[t][i >> 1] | (v << 8);
    }
  }
  int* const B = p.B + (size_t)((k0 >> 4) + (chunk >> 1)) * 2 * p.n + blk * 128 + 16 * (lane >> 3) + 8 * odd;
#pragma unroll
  for (int x = 0; x < 2; x++) {
    i4 out;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int got = __shfl_xor(odd ? half[x][j] : half[2 + x][j], 1);
      out[j] = odd ? got | (half[2 + x][j] << 4) : half[x][j] | (got << 4);
    }
    *(i4*)(B + 4 * x) = out;
  }
}

thread_local char g_convert_error[256] = "";

// `dev` current for the length of a call
struct OnDevice {
  int prev = -1;
  hipError_t e;
  explicit OnDevice(int dev) {
    e = hipGetDevice(&prev);
    if (e == hipSuccess && prev != dev) e = hipSetDevice(dev);
    else prev = -1;
    (void)hipGetLastError();  // an earlier call's error is not this launch's
  }
  int done() {
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) return MARLIN_OK;
    snprintf(g_convert_error, sizeof(g_convert_error), "%s", hipGetErrorString(e));
    return MARLIN_ERR_RUNTIME;
  }
  ~OnDevice() {
    if (prev >= 0) (void)hipSetDevice(prev);
  }
};

// a launch has at most 65535 rows of workgroups and 2^32 - 1 threads in a row
bool grid_holds(long long x, int threads, long long y) {
  return x * threads <= 0xffffffffLL && y <= 65535;
}
long long pieces_of(long long a, int b) { return (a + b - 1) / b; }

// Whether long groups are quantised in chunks, on a device of `cus` compute units.  In
// one launch, a workgroup per group of 64 columns, a row takes a round of workgroups 14
// to 30 ns, however few they are; in chunks the chip is full whatever n is, but w is
// read twice and there are three launches.  One scale per column, 256 compute units, us
// in one launch and in chunks: n = 1024, k = 1024 15.6 and 15.6, 2048 28.7 and 16.2, 8192
// 113.7 and 22.5; n = 4096 1024 17.1 and 17.6, 4096 74.9 and 31.4, 8192 156 and 58; n =
// 8192 2048 40.4 and 30.3; n = 11008 1024 23.9 and 24.2, 4096 100.8 and 82.0; n = 16384
// 2048 52.0 and 64.9, 4096 120.8 and 127.3; n = 28672 1024 46.6 and 49.7, 8192 556 and
// 454.
bool in_chunks(int n, int k, int gs, int cus) {
  const long long wgs = pieces_of(n, 64) * (k / gs);
  const double rounds = (double)pieces_of(wgs, cus);
  const double whole = gs * rounds * (0.0139 + 6.1e-5 * (wgs < cus ? wgs : cus));
  const double chunks = 16.0 + gs * wgs * 1.02e-4;
  return chunks < whole && pieces_of(gs, kChunkRows) * (k / gs) <= 65535;
}

bool aligned(const void* p) { return ((uintptr_t)p & 15) == 0; }

bool apart(const void* a, size_t a_bytes, const void* b, size_t b_bytes) {
  return (uintptr_t)a + a_bytes <= (uintptr_t)b || (uintptr_t)b + b_bytes <= (uintptr_t)a;
}

}  // namespace

}  // namespace w4a16

using namespace w4a16;

extern "C" {

int marlin_amd_quantize(const void* w, int k, int n, int groupsize, int by_column, void* fake,
                        void* q, void* s, int dev, void* stream) {
  const int gs = groupsize == -1 ? k : groupsize;
  if (k <= 0 || n <= 0 || gs <= 0 || k % gs != 0 || (by_column ? gs : n) % 4 != 0 ||
      !aligned(w) || !aligned(fake) || !aligned(q) || !aligned(s))
    return MARLIN_ERR_PROB_SHAPE;
  const long long teams = (long long)n * (k / gs);
  const bool small = gs <= 128;
  if (by_column ? !grid_holds(small ? pieces_of(teams, 8) : teams, kPThreads, 1)
                : !grid_holds(pieces_of(n, small ? 256 : 64), kQThreads, k / gs))
    return MARLIN_ERR_PROB_SHAPE;
  OnDevice on(dev);
  int cus = 0;
  if (on.e == hipSuccess && !by_column && !small)
    on.e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (on.e != hipSuccess) return on.done();
  const half_t* in = (const half_t*)w;
  const hipStream_t st = (hipStream_t)stream;
  if (by_column) {
    if (small)
      hipLaunchKernelGGL(quantise_columns<32>, dim3((unsigned)pieces_of(teams, 8)), dim3(kPThreads), 0,
                         st, in, n, k, gs, (half_t*)fake, (int*)q, (half_t*)s);
    else
      hipLaunchKernelGGL(quantise_columns<kPThreads>, dim3((unsigned)teams), dim3(kPThreads), 0, st,
                         in, n, k, gs, (half_t*)fake, (int*)q, (half_t*)s);
  } else if (small) {
    hipLaunchKernelGGL(quantise_rows<64>, dim3((unsigned)pieces_of(n, 256), k / gs), dim3(kQThreads), 0, st, in,
                       n, gs, (half_t*)fake, (int*)q, (half_t*)s);
  } else if (in_chunks(n, k, gs, cus)) {
    const int per_group = (int)pieces_of(gs, kChunkRows);
    const dim3 chunks((unsigned)pieces_of(n, 256), (unsigned)(k / gs) * per_group);
    hipLaunchKernelGGL(chunk_maxima, chunks, dim3(kQThreads), 0, st, in, n, gs, per_group, (unsigned short*)q);
    hipLaunchKernelGGL(chunk_scales, dim3((unsigned)pieces_of(n, 64), k / gs), dim3(kQThreads), 0, st,
                       (const unsigned short*)q, n, per_group, (half_t*)s);
    hipLaunchKernelGGL(quantise_chunks, chunks, dim3(kQThreads), 0, st, in, n, gs, per_group, (half_t*)fake,
                       (int*)q, (const half_t*)s);
  } else {
    hipLaunchKernelGGL(quantise_rows<16>, dim3((unsigned)pieces_of(n, 64), k / gs), dim3(kQThreads), 0, st, in, n,
                       gs, (half_t*)fake, (int*)q, (half_t*)s);
  }
  return on.done();
}

int marlin_amd_quantize_launches(int k, int n, int groupsize, int by_column, int cus) {
  const int gs = groupsize == -1 ? k : groupsize;
  if (k <= 0 || n <= 0 || gs <= 0 || k % gs != 0 || cus <= 0) return 0;
  return !by_column && gs > 128 && in_chunks(n, k, gs, cus) ? 3 : 1;
}

int marlin_amd_pack(const void* w, int k, int n, int groupsize, int by_column, const void* scales,
                    long long s_group, long long s_col, void* B, void* s_packed, int dev,
                    void* stream) {
  const int gs = groupsize == -1 ? k : groupsize;
  if (k <= 0 || n <= 0 || gs <= 0 || n % 64 != 0 || k % 64 != 0 || gs % 64 != 0 || k % gs != 0 ||
      !aligned(w) || !aligned(B) || s_group < 0 || s_col < 0 ||
      (by_column ? !grid_holds(n / 64, kPThreads, pieces_of(k, 256))
                 : !grid_holds(pieces_of(n, 2 * kPThreads), kPThreads, k / 16)))
    return MARLIN_ERR_PROB_SHAPE;
  // every workgroup reads scales while others write packed ones
  const int groups = k / gs;
  const size_t w_bytes = (size_t)k * n * 2, b_bytes = (size_t)k * n / 2, p_bytes = (size_t)groups * n * 2;
  const size_t s_bytes = (size_t)((groups - 1) * s_group + (n - 1) * s_col + 1) * 2;
  if (!apart(B, b_bytes, w, w_bytes) || !apart(B, b_bytes, scales, s_bytes) ||
      !apart(B, b_bytes, s_packed, p_bytes) || !apart(s_packed, p_bytes, w, w_bytes) ||
      !apart(s_packed, p_bytes, scales, s_bytes))
    return MARLIN_ERR_PROB_SHAPE;
  OnDevice on(dev);
  if (on.e != hipSuccess) return on.done();
  const PackArgs p = {w, (const half_t*)scales, s_group, s_col, (int*)B, (half_t*)s_packed,
                      k, n, gs, groupsize != -1};
  if (by_column)
    hipLaunchKernelGGL(pack_columns, dim3(n / 64, (unsigned)pieces_of(k, 256)), dim3(kPThreads), 0,
                       (hipStream_t)stream, p);
  else
    hipLaunchKernelGGL(pack_rows<false>, dim3((unsigned)pieces_of(n, 2 * kPThreads), k / 16), dim3(kPThreads), 0,
                       (hipStream_t)stream, p);
  return on.done();
}

int marlin_amd_pack_words(const void* q, int k, int n, void* B, int dev, void* stream) {
  if (k <= 0 || n <= 0 || n % 64 != 0 || k % 16 != 0 || !aligned(q) || !aligned(B) ||
      !grid_holds(pieces_of(n, 2 * kPThreads), kPThreads, k / 16))
    return MARLIN_ERR_PROB_SHAPE;
  OnDevice on(dev);
  if (on.e != hipSuccess) return on.done();
  const PackArgs p = {q, nullptr, 0, 0, (int*)B, nullptr, k, n, k, false};
  hipLaunchKernelGGL(pack_rows<true>, dim3((unsigned)pieces_of(n, 2 * kPThreads), k / 16), dim3(kPThreads), 0,
                     (hipStream_t)stream, p);
  return on.done();
}

const char* marlin_amd_convert_last_error(void) { return g_convert_error; }

}  // extern "C"
