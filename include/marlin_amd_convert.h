/*
 * Weight conversion of libmarlin_amd.so: fp16 weights to 4 bits and to the
 * packed layout that marlin_gemm reads, on the GPU.  The layouts are those of
 * the reference's Layer.pack (gemm/marlin_gemm/marlin.py:92-131), the
 * quantiser that of its tests (marlin_test.py:18-40); both are tensor
 * arithmetic there and have no entry in its binding.
 *
 * All pointers are device pointers, fp16 weights and scales, 16-byte aligned.
 * Calls are asynchronous on `stream` and need no workspace.  Returns one of
 * marlin_gemm's codes; MARLIN_ERR_PROB_SHAPE also for a problem that no grid
 * holds (some hundred million groups, a million rows).
 */
#ifndef MARLIN_AMD_CONVERT_H
#define MARLIN_AMD_CONVERT_H

#include "marlin_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * Symmetric 4-bit quantisation: per column and group of `groupsize` k-values
 * (-1: all of k) s = fp16(max|w| * 2/15), q = clamp(round(fp16(w / s)) + 8, 0,
 * 15), fake = fp16((q - 8) * s).
 * by_column = 0: w, fake (fp16) and q (int32) are (k, n) with the columns
 * contiguous, n a multiple of 4; by_column = 1: the same values stored column
 * by column, i.e. as (n, k), groupsize a multiple of 4.  s: (groups, n) fp16.
 * (Where groups are long, q holds intermediate values before its own.)
 */
int marlin_amd_quantize(const void *w, int k, int n, int groupsize, int by_column, void *fake,
                        void *q, void *s, int dev, void *stream);

/*
 * Fake-quantised weights and their scales to packed words and packed scales:
 * q = clamp(round(fp16(w / s)) + 8, 0, 15).  w as above, n a multiple of 64, k
 * of 64; scale of group g and column c at scales[g * s_group + c * s_col];
 * groupsize -1 or a multiple of 64, no stride negative.  B: (k/16, 2n) int32;
 * s_packed: (groups, n) fp16; neither may overlap the other, w or scales.
 */
int marlin_amd_pack(const void *w, int k, int n, int groupsize, int by_column, const void *scales,
                    long long s_group, long long s_col, void *B, void *s_packed, int dev,
                    void *stream);

/* Whole numbers in [0, 15], (k, n) int32 with k a multiple of 16 and n of 64,
 * to packed words. */
int marlin_amd_pack_words(const void *q, int k, int n, void *B, int dev, void *stream);

/* Text of the calling thread's last MARLIN_ERR_RUNTIME from this header. */
const char *marlin_amd_convert_last_error(void);

#ifdef __cplusplus
}
#endif
#endif
