/* SPDX-License-Identifier: MPL-2.0
 *
 * rows_gemm.h — the plain matmul over unquantized rows for several input rows (rows_gemm.hip).
 */
#ifndef BMK_ROWS_GEMM_H
#define BMK_ROWS_GEMM_H

#include <hip/hip_runtime.h>

enum { RG_F32 = 0, RG_BF16 = 2, RG_F16 = 3 }; /* weight formats, as the LM head's */

#ifdef __cplusplus
extern "C" {
#endif
/* whether the shape (weights in format wf) is better served by rows_gemm_launch */
int rows_gemm_ok(int BT, int C, int OC, int wf);
/* out[BT][OC] = x[BT][C] x w^T (+ bias); x and w 4-byte aligned, C a multiple of 32; -1: refused */
int rows_gemm_launch(const float* x, const void* w, int wf, const float* bias, float* out, int BT, int C, int OC,
                     hipStream_t s);
#ifdef __cplusplus
}
#endif

#endif
