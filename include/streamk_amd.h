/* C ABI of the dense fp16 GEMM with a stream-K tail in libmarlin_amd.so (gfx950).
 *
 * The reference's gemm/streamk_gemm is a stand-alone program without a library
 * interface: gemm_streamk.cu:8-110 builds A (m x k, row-major), B (k x n,
 * column-major, i.e. n rows of k) and C (m x n, row-major) in fp16 with
 * alpha = 1, beta = 0, fills an Arguments object (gemm_streamk.h, with the tile
 * split of dp_sk_block.h:31-128), allocates its workspace (init_workspace) and
 * launches gemmTN_streamk_dp.  streamk_gemm_tn stands for that sequence: the
 * caller passes the three device buffers and the sizes; the split, the
 * workspace and the launch are the library's.
 */
#ifndef STREAMK_AMD_H
#define STREAMK_AMD_H

#ifdef __cplusplus
extern "C" {
#endif

#define STREAMK_OK 0
#define STREAMK_ERR_SHAPE 1   /* negative size, n not a multiple of 256, k not a multiple of 64 */
#define STREAMK_ERR_RUNTIME 3 /* HIP error or size limit; text in streamk_amd_last_error() */

/* C = A * B^T on `hip_stream` (a hipStream_t) of device `dev`; asynchronous.
 * A: m x k fp16, row-major.  B: n x k fp16, row-major (the k x n column-major
 * operand of gemm_streamk.cu:29).  C: m x n fp16, row-major, written once.
 * fp32 accumulation.  m is arbitrary; n % 256 == 0 and k % 64 == 0.
 * Partial sums of the stream-K tiles live in the library-owned buffer of this
 * (device, stream) that marlin_gemm uses too (include/marlin_amd.h): sized by
 * the launch (64 KiB per slice of a 128 x 128 tile, 128 KiB of a 128 x 256
 * one), grown on demand, none for launches without slices.  Calls on one stream
 * may follow each other freely, calls that overlap must use different streams; a
 * call that would have to allocate under graph capture returns
 * STREAMK_ERR_RUNTIME.  What the launch is (slices or whole tiles, see below)
 * may depend on the capture and on the scratch, the bits of C do not. */
int streamk_gemm_tn(const void* A, const void* B, void* C, int m, int n, int k, int dev,
                    void* hip_stream);

/* return code streamk_gemm_tn would give for these sizes (no GPU touched) */
int streamk_amd_check(int m, int n, int k);

/* the tile split for a device with `cus` compute units (counterpart of
 * SK_DP_Block_Wrapper, dp_sk_block.h:31-80): out[0..7] = tiles along m, tiles
 * along n (tiles numbered in panels of 8 column tiles), data-parallel tiles, stream-K
 * tiles (the last ones in tile order), k slices per stream-K tile, (tile, slice)
 * pairs, rows of a tile (256, or 128 when 256 x 256 tiles would occupy at most
 * half of the compute units), columns of a tile (256, or 128 when 128 x 256 tiles
 * would occupy at most half of them too).  streamk_amd_launches and
 * streamk_amd_tile say how the problem is computed. */
int streamk_amd_plan(int m, int n, int k, int cus, int* out);

/* out[0..2] = rows, columns and k slices of the tiles, 32 x 32 to 128 x 256, that
 * compute the problem in one launch of a workgroup per tile and slice, in place of
 * streamk_amd_launches, where they fill the compute units better; zeros where they
 * do not.  Returns what streamk_amd_check does. */
int streamk_amd_tile(int m, int n, int k, int cus, int* out);

/* such tiles for every problem of the calling thread, whatever their cost, in at
 * most the plan's slices: rows = 0 back to the choice by cost, < 0 never; for tests
 * and tools */
void streamk_amd_force_tile(int rows, int cols, int slices);

/* the launches that compute the plan's tiles, at most two, five numbers each: rows and
 * columns of a workgroup's tile, waves of a workgroup, tiles, slices of the k
 * range per tile (a workgroup per tile and slice).  The stream-K tiles of 256 x 256
 * are computed as four 128 x 128 quarters each, in as many slices as leave none
 * without a compute unit; and from k = 7168, with scratch != 0, two neighbouring
 * whole 128 x 128 tiles as two slices of a 128 x 256 one (a call under capture,
 * or whose scratch cannot be had, goes without).  Returns their number; 0 for
 * sizes that are refused or empty. */
int streamk_amd_launches(int m, int n, int k, int cus, int scratch, int* out);

/* out[0], out[1] = row and column tile of tile number `tile` (0 <= tile <
 * tiles_m * tiles_n); for tests of the numbering */
void streamk_amd_tile_coord(int tile, int tiles_m, int tiles_n, int* out);

/* (tile, slice) that workgroup `block` of a launch of tiles * slices workgroups
 * computes; for tests of the order */
void streamk_amd_slice_coord(int block, int tiles, int slices, int* out);

/* how often a workgroup looks whether the other slices of its tile have arrived
 * before it leaves them its share of the sums, for the calling thread: -1 = the
 * default, 0 = at once; for tests (results do not depend on it) */
void streamk_amd_force_finish_polls(int polls);

/* same as marlin_amd_release (include/marlin_amd.h): frees the partial-sum
 * buffers of device dev (all if dev < 0), returns the bytes freed */
long long streamk_amd_release(int dev);

/* text of the last STREAMK_ERR_RUNTIME on this thread */
const char* streamk_amd_last_error(void);

#ifdef __cplusplus
}
#endif
#endif
