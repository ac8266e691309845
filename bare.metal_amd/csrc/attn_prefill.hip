/* SPDX-License-Identifier: MPL-2.0
 *
 * attn_prefill.hip — causal attention of a whole prompt, head size 64, on fp32 MFMA
 * (v_mfma_f32_16x16x4f32): softmax(q.k * scale) over keys 0..p times V, for
 * every position p of every query head.  Two sources share the kernel:
 *  - AP_ENGINE: the engine's prefill.  q rows roped [n][NH*64], K and V from
 *    a layer's KV cache (K per KV head as [16][MS] float4, V row-major
 *    [MS][KV]), output bf16 in fragment order (the o projection's operand).
 *  - AP_FLAT: the reference's prefill attention ABI (forward.metal:1904-2114):
 *    Q roped [S][NH][64], K and V [S][NKV][64], fp32 output [S][NH][64].
 *
 * A workgroup takes 16 consecutive positions of one head; its waves take the
 * 16-key sub-blocks up to the diagonal in turn.  Per sub-block a wave forms
 *   S^T (16 keys x 16 queries) = K_sb Q^T   (16 MFMAs over the 64 dims),
 * updates a per-query online softmax, and accumulates
 *   O^T (64 dims x 16 queries) += V_sb^T P^T (16 MFMAs).
 * The MFMA sums run over any order of their index, so both products use a
 * permuted one: in S^T, step s of lane group g (= lane/16) takes dimension
 * 16g + s (a lane holds 16 consecutive dims of its key); in O^T, step s of
 * lane group g takes key 4g + s, which is exactly the key whose score that
 * lane holds in element s of its S^T fragment, so P^T goes from the score
 * registers to the next MFMA with no data movement.  Each wave's (max, sum,
 * O^T) is merged across waves through LDS at the end.
 *
 * What bounds it: the matrix pipe's fp32 rate for long prompts (a sub-block
 * is 1024 cycles of one SIMD's), the chain of sub-blocks of the longest
 * block for short ones.  No element of K or V is used by two waves, so
 * nothing is staged for a workgroup and no barrier runs in the loop (the form
 * before staged 128-key chunks through LDS for 8 waves): a wave loads its
 * next two sub-blocks into registers, V straight as MFMA operands (64-byte
 * runs), K straight from the engine's cache layout and, from rows, through
 * 8 KB of LDS that only it uses.  The running maximum is moved only when a
 * score passes it by 2^8, so the reduction over the lane groups and the
 * rescaling of O are rare; sums stay far inside fp32's range and their
 * relative error is the same.  A wave's two sub-blocks of a turn are summed
 * on their own before they join O: with four waves the products straight into
 * O are chains twice as long as with eight, and the error against 64 bits grew
 * with the prompt (N(0, 1), 512 / 2048 / 4096 positions, 1e-7: eight waves 1.48 /
 * 1.83 / 2.15, four 1.56 / 2.11 / 2.60, so 1.45 / 1.61 / 1.70).
 * GPU time per launch, back to back, before / now, 15 heads on 5 KV heads: 16
 * positions 6.1 / 4.4 us, 333 14.1 / 10.0, 512 21.9 / 14.0, 1024 61.2 / 32.7, 2048 198 / 92
 * (the products alone take 52); 9 heads on 3, 512 positions: 15.8 / 11.6; the
 * turns' own sums cost up to 4% of that (2048: 98.35 -> 98.43, kernel trace).  8 waves
 * per workgroup: 104 us at 2048, 5.8 at 16; one sub-block at a time: the same
 * within 2%; a register budget for 4 waves per SIMD spills (193 us).
 */
#include "bmk.h"
#include "attn_prefill.h"
#include "q8_common.h"

#include <math.h>

namespace {

using namespace bmk;

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int QB = 16;     /* positions per workgroup */
constexpr int AW = 4;      /* waves per workgroup */
constexpr int HD = 64;
constexpr float SLACK = 8.0f; /* in powers of two */
enum { AP_ENGINE = 0, AP_FLAT = 1 };

__device__ __forceinline__ f32x4 ld4(const float* p) {
    f32x4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 16), 16);
    return v;
}

template <int MODE>
__global__ __launch_bounds__(64 * AW) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_attn_prefill(ApArgs a) {
    __shared__ __attribute__((aligned(16))) float Ws[AW * 2 * 16 * HD]; /* K staging, 32 keys a wave; then the merge */
    __shared__ float Ms[AW * QB], Ls[AW * QB];
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const int col = lane & 15, grp = lane >> 4; /* MFMA column (query / key row) and lane group */
    /* the last blocks of the prompt have the most keys: they take the first
     * workgroup slots, and the short ones fill in behind them (measured: the
     * heads dealt to the XCDs in whole, for their L2s, leaves CUs idle at the
     * end, 512 positions 11.6 -> 15.4 us, 2048 and 15 heads 92 -> 109) */
    const int h = blockIdx.x, p0 = (int)(gridDim.y - 1 - blockIdx.y) * QB;
    const int kh = h / a.kv_mul, n = a.n;
    const int p = p0 + col; /* this lane's query position */
    const float sl2 = a.scale * 1.44269504088896341f; /* scores in base 2 */
    const int nsb = (min(p0 + QB, n) + 15) >> 4;
    const float* kb = a.k + (MODE == AP_FLAT ? (size_t)kh * HD : (size_t)kh * HD * a.MS);
    const float* vb = a.v + (size_t)kh * HD;

    /* a sub-block's rows from a wave-uniform base and fixed 32-bit lane offsets (bytes) */
    unsigned int ko[4], vo[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        ko[i] = 4u * (MODE == AP_FLAT ? (unsigned)((4 * i + grp) * a.KV + 4 * col)
                                      : (unsigned)((4 * grp + i) * a.MS + col) * 4u);
        vo[i] = 4u * (unsigned)((4 * grp + i) * a.KV + col);
    }
    /* keys at or past n (the prompt's last sub-block) read row n - 1; past the last sub-block the loads repeat it */
    auto fetch_k = [&](int sb, f32x4* k) {
        const int k0 = 16 * min(sb, nsb - 1), last = n - 1 - k0;
        const char* ks = (const char*)(kb + (size_t)k0 * (MODE == AP_FLAT ? a.KV : 4));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const unsigned int past = 4u * (MODE == AP_FLAT ? (unsigned)(last * a.KV + 4 * col)
                                                            : (unsigned)((4 * grp + i) * a.MS + last) * 4u);
            k[i] = ld4((const float*)(ks + ((MODE == AP_FLAT ? 4 * i + grp : col) <= last ? ko[i] : past)));
        }
    };
    auto fetch_v = [&](int sb, float* v) {
        const int k0 = 16 * min(sb, nsb - 1), last = n - 1 - k0;
        const char* vs = (const char*)(vb + (size_t)k0 * a.KV);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const unsigned int o = 4 * grp + i <= last ? vo[i] : 4u * (unsigned)(last * a.KV + col);
#pragma unroll
            for (int d = 0; d < 4; d++) v[4 * i + d] = *(const float*)(vs + o + 64 * d);
        }
    };
    /* Q^T fragment: step s holds q[col][16*grp + s] */
    f32x4 qf[4];
    {
        const float* qr = a.q + ((size_t)min(p, n - 1) * a.NH + h) * HD + 16 * grp;
#pragma unroll
        for (int i = 0; i < 4; i++) qf[i] = ld4(qr + 4 * i);
    }
    f32x4 k0r[4], k1r[4];
    float v0r[16], v1r[16];
    /* loads in this order on both ways into the loop, or its waits are for the worse */
    __builtin_amdgcn_sched_barrier(0);
    fetch_k(wave, k0r);
    fetch_k(wave + AW, k1r);
    __builtin_amdgcn_sched_barrier(0);
    fetch_v(wave, v0r);
    fetch_v(wave + AW, v1r);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc[4]; /* O^T tile d: dims 16d + 4*grp + v, query col */
    auto zero = [](f32x4* o) {
#pragma unroll
        for (int d = 0; d < 4; d++) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    zero(acc);
    float m = -INFINITY, l = 0.0f; /* m: per query (same in the 4 lane groups); l: this lane's keys */

    /* S^T[key 4*grp + v][query col] of a sub-block, times scale * log2(e) */
    auto scores = [&](const f32x4* k, float* Kw) {
        f32x4 kf[4];
        if (MODE == AP_FLAT) {
            /* rows to lanes through this wave's LDS (one wave: in order, no
             * barrier); key r's 16-byte chunk c sits at c ^ r, so that the 16
             * keys a chunk is read from fall in different banks */
#pragma unroll
            for (int i = 0; i < 4; i++) *(f32x4*)&Kw[(4 * i + grp) * HD + 4 * (col ^ (4 * i + grp))] = k[i];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 4; i++) kf[i] = *(const f32x4*)&Kw[col * HD + 4 * ((4 * grp + i) ^ col)];
            __builtin_amdgcn_wave_barrier();
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) kf[i] = k[i];
        }
        /* four independent chains over the 64 dimensions (a single chain waits out each MFMA's latency) */
        f32x4 sq[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sq[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            sq[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i].x, qf[i].x, sq[i], 0, 0, 0);
        }
#pragma unroll
        for (int e = 1; e < 4; e++)
#pragma unroll
            for (int i = 0; i < 4; i++) sq[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][e], qf[i][e], sq[i], 0, 0, 0);
        return ((sq[0] + sq[1]) + (sq[2] + sq[3])) * sl2;
    };
    auto max4 = [](const f32x4& v) { return fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)); };
    auto move_max = [&](float cm) { /* cm: this lane's largest new score */
        if (__any(cm > m + SLACK)) { /* also the first score of any query (m = -inf) */
            cm = fmaxf(cm, __shfl_xor(cm, 16));
            cm = fmaxf(cm, __shfl_xor(cm, 32));
            const float mn = fmaxf(m, cm);
            const float fr = mn > -INFINITY ? __builtin_amdgcn_exp2f(m - mn) : 1.0f;
            l *= fr;
#pragma unroll
            for (int d = 0; d < 4; d++) acc[d] *= fr;
            m = mn;
        }
    };
    auto weights = [&](const f32x4& sv) {
        f32x4 pv;
#pragma unroll
        for (int v = 0; v < 4; v++) pv[v] = m > -INFINITY ? __builtin_amdgcn_exp2f(sv[v] - m) : 0.0f;
        return pv;
    };
    auto sum4 = [](const f32x4& v) { return (v.x + v.y) + (v.z + v.w); };
    /* O^T[dim 16d + col'][query] += V^T[dim][key 4*grp + i] * P^T[key][query] */
    auto values = [&](const float* v, const f32x4& pv, f32x4* o) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int d = 0; d < 4; d++) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[4 * i + d], pv[i], o[d], 0, 0, 0);
    };
    auto add = [&](const f32x4* o) {
#pragma unroll
        for (int d = 0; d < 4; d++) acc[d] += o[d];
    };
    float* Kw = &Ws[wave * 2 * 16 * HD];
    /* Below the diagonal two sub-blocks at a time, so that one's products run
     * beside the other's softmax.  K's next rows are loaded behind its
     * products, V's behind theirs, into the registers just read (the
     * scheduler, left alone, loads into others and copies, which waits for
     * the loads; a branch around a load does the same). */
    int sb = wave;
    for (; sb + AW < nsb - 1; sb += 2 * AW) {
        const f32x4 sa = scores(k0r, Kw), sc = scores(k1r, Kw + 16 * HD);
        __builtin_amdgcn_sched_barrier(0);
        fetch_k(sb + 2 * AW, k0r);
        fetch_k(sb + 3 * AW, k1r);
        __builtin_amdgcn_sched_barrier(0);
        move_max(fmaxf(max4(sa), max4(sc)));
        f32x4 o2[4]; /* a turn's own sum first: acc's chain has one rounding per 32 keys of the wave instead of eight */
        zero(o2);
        const f32x4 pa = weights(sa);
        values(v0r, pa, o2);
        const f32x4 pc = weights(sc);
        values(v1r, pc, o2);
        l += sum4(pa) + sum4(pc);
        add(o2);
        __builtin_amdgcn_sched_barrier(0);
        fetch_v(sb + 2 * AW, v0r);
        fetch_v(sb + 3 * AW, v1r);
        __builtin_amdgcn_sched_barrier(0);
    }
    /* the last one or two, the diagonal's among them (sub-block nsb - 1) */
    auto last_one = [&](int sb, const f32x4* k, const float* v) {
        f32x4 sv = scores(k, Kw);
        float vz[16];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int key = 16 * sb + 4 * grp + i;
            sv[i] = key <= p ? sv[i] : -INFINITY;
#pragma unroll
            for (int d = 0; d < 4; d++) vz[4 * i + d] = key < n ? v[4 * i + d] : 0.0f; /* past n there is nothing */
        }
        move_max(max4(sv));
        f32x4 o2[4];
        zero(o2);
        const f32x4 pv = weights(sv);
        l += sum4(pv);
        values(vz, pv, o2);
        add(o2);
    };
    if (sb < nsb) last_one(sb, k0r, v0r);
    if (sb + AW < nsb) last_one(sb + AW, k1r, v1r);
    /* this wave's sum over its keys: add the four lane groups */
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    __syncthreads(); /* the merge lies over other waves' K staging */
    /* [wave][dim][query] */
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int v = 0; v < 4; v++) Ws[(wave * HD + 16 * d + 4 * grp + v) * QB + col] = acc[d][v];
    if (grp == 0) {
        Ms[wave * QB + col] = m;
        Ls[wave * QB + col] = l;
    }
    __syncthreads();
    const int r = t >> 4, g = t & 15; /* query r, dimensions 4g .. 4g+3 */
    static_assert(64 * AW >= QB * HD / 4, "a thread per four outputs");
    if (r >= QB || p0 + r >= n) return;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < AW; w++) mx = fmaxf(mx, Ms[w * QB + r]);
    float den = 0.f, o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;
#pragma unroll
    for (int w = 0; w < AW; w++) {
        const float mv = Ms[w * QB + r];
        const float fr = mv == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mv - mx);
        const float* src = &Ws[(w * HD + 4 * g) * QB + r];
        den = fmaf(fr, Ls[w * QB + r], den);
        o0 = fmaf(fr, src[0 * QB], o0);
        o1 = fmaf(fr, src[1 * QB], o1);
        o2 = fmaf(fr, src[2 * QB], o2);
        o3 = fmaf(fr, src[3 * QB], o3);
    }
    if (MODE == AP_FLAT) {
        *(f32x4*)&a.out[((size_t)(p0 + r) * a.NH + h) * HD + 4 * g] = f32x4{o0 / den, o1 / den, o2 / den, o3 / den};
    } else { /* the o projection's operand: fragment order, four consecutive values */
        const uint2 o = make_uint2((unsigned int)bf16_bits(o0 / den) | ((unsigned int)bf16_bits(o1 / den) << 16),
                                   (unsigned int)bf16_bits(o2 / den) | ((unsigned int)bf16_bits(o3 / den) << 16));
        *(uint2*)(a.out16 + frag_index(p0 + r, h * HD + 4 * g, a.NH)) = o;
    }
}

} // namespace

extern "C" int ap_launch(const ApArgs* a, int engine, hipStream_t s) {
    const dim3 grid(a->NH, (a->n + QB - 1) / QB);
    if (engine) hipLaunchKernelGGL(k_attn_prefill<AP_ENGINE>, grid, dim3(64 * AW), 0, s, *a);
    else hipLaunchKernelGGL(k_attn_prefill<AP_FLAT>, grid, dim3(64 * AW), 0, s, *a);
    BMK_LAUNCH_CHECK();
    return 0;
}
