/* SPDX-License-Identifier: MPL-2.0
 *
 * attn_prefill.h — causal attention of a prompt, head size 64 (attn_prefill.hip).
 */
#ifndef BMK_ATTN_PREFILL_H
#define BMK_ATTN_PREFILL_H

#include <hip/hip_runtime.h>

typedef struct {
    const float* q;        /* [n][NH][64], roped, 16-byte aligned */
    const float* k;        /* flat: [n][KV] rows; engine: the layer's K cache, [KV head][16][MS] float4 */
    const float* v;        /* rows of KV floats */
    float* out;            /* flat: [n][NH][64], 16-byte aligned */
    unsigned short* out16; /* engine: bf16 [n][NH*64] in fragment order */
    int NH, n, kv_mul, KV, MS;
    float scale;
} ApArgs;

#ifdef __cplusplus
extern "C" {
#endif
int ap_launch(const ApArgs* a, int engine, hipStream_t s);
#ifdef __cplusplus
}
#endif

#endif
