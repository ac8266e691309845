/* SPDX-License-Identifier: MPL-2.0
 *
 * attn_decode.hip — attention_forward, one query position over the KV cache
 * in the reference's row layout (reference src/kernels/forward.metal:1362-1465):
 *   out[h] = softmax(scale * q[h].K[0..S-1]) V[0..S-1], fp32, head h on KV head h / kv_mul.
 *
 * What bounds it: bytes in flight.  One layer's K and V are 5 MB at
 * SmolLM2-360M and 2048 keys, 1 us of HBM time, so one workgroup per query
 * head (15 workgroups walking all keys in turn) is a latency chain on a
 * nearly idle chip.  Here a workgroup takes one split of the keys of one KV
 * head and, past two tiles of keys, serves up to four of its query heads, so
 * every K and V row is read once per four heads, and all of a tile's loads
 * are issued before the first is used.  The last workgroup of a KV head to
 * finish merges the splits' (max, sum, partial output) records.
 *
 * GPU time per launch, back to back, 15 query heads on 5 KV heads of 64, one
 * workgroup per head before / splits now: 301 keys 17.4 (9 heads on 3) / 6.6 us,
 * 2048 keys 155 / 7.5 us, 4096 keys 10.3 us; one key takes 3.2 us, two
 * tiles 3.9 us (kernel trace).  What is left is latency: loads, two handovers, the merge.  With 8
 * waves of 16 keys instead of 4: 0.2-0.9 us more up to 2048 keys, 1.6 us less
 * at 4096.  The merge reads at most 16 records of an output at once: 32
 * measured 0.3 us slower up to 1000 keys, and reading a clamped record again
 * instead of none past the last one took a launch to 19 us (every lane of every
 * head then reads the same lines past the L2).
 */
#include "bmk.h"
#include "q8_common.h"

#include <math.h>

#include <algorithm>

namespace {

using namespace bmk;

constexpr int AT_WAVES = 4, AT_NT = 64 * AT_WAVES;
constexpr int AT_MAX_SPLIT = 64; /* records the merge holds weights for in LDS */
/* The scratch memory starts with the arrival counters, each on a line of its
 * own (same-line atomics queue up); records never overwrite that part, so
 * the counters stay zero between launches of any shape. */
constexpr int AT_DONE_STRIDE = 32, AT_MAX_GROUPS = 1024;
constexpr size_t AT_DONE_BYTES = (size_t)AT_DONE_STRIDE * AT_MAX_GROUPS * 4;

/* Keys a wave takes per tile: each load instruction covers 256 / HD keys (16
 * bytes a lane), AT_UN of them in flight for K and for V. */
template <int HD> struct AtTile {
    static constexpr int LPK = HD / 4;   /* lanes per key row */
    static constexpr int KPI = 64 / LPK; /* keys per load instruction */
    static constexpr int UN = HD <= 64 ? 4 : 8;
    static constexpr int WKEYS = KPI * UN;
    static constexpr int KEYS = AT_WAVES * WKEYS;
};

struct AtArgs {
    const float* q;
    const float* k; /* the layer's K rows, [MS][KV] */
    const float* v;
    float* out;
    float* rec;         /* [group][split][QH][HD + 2]: partial output, max, sum */
    unsigned int* done; /* [group * AT_DONE_STRIDE] workgroups arrived; zero between launches */
    int NH, KV, S, kv_mul, ng; /* ng: workgroup groups per KV head */
    int keys, nsplit;          /* keys per split, a multiple of the tile */
    float scale;
};

__device__ __forceinline__ float agent_load(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* weight of a partial with maximum m beside the common maximum M; a partial
 * without a finite score (m = -inf) has nothing but what its sum says */
__device__ __forceinline__ float at_weight(float m, float M) { return m == -INFINITY ? 0.0f : expf(m - M); }

/* Sum over LPK consecutive lanes (every one gets it): within 16 lanes by DPP,
 * beyond by shuffles. */
template <int CTRL>
__device__ __forceinline__ float at_dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
template <int LPK>
__device__ __forceinline__ float row_sum(float v) {
    if (LPK >= 2) v += at_dpp<0xB1>(v);  /* quad_perm: lane ^ 1 */
    if (LPK >= 4) v += at_dpp<0x4E>(v);  /* quad_perm: lane ^ 2 */
    if (LPK >= 8) v += at_dpp<0x141>(v); /* row_half_mirror: the other quad of 8 */
    if (LPK >= 16) v += at_dpp<0x140>(v); /* row_mirror: the other half of 16 */
    if (LPK >= 32) v += __shfl_xor(v, 16);
    if (LPK >= 64) v += __shfl_xor(v, 32);
    return v;
}

template <int HD, int QH>
__global__ __launch_bounds__(AT_NT) void k_attn_decode(AtArgs a) {
    typedef AtTile<HD> T;
    constexpr int LPK = T::LPK, UN = T::UN;
    constexpr int REC = HD + 2;
    __shared__ float wacc[AT_WAVES][QH][HD];
    __shared__ float wm[AT_WAVES][QH], wl[AT_WAVES][QH];
    __shared__ float rf[QH][64], rl[QH]; /* the merge: records' weights, sums */
    __shared__ int last;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int nsplit = a.nsplit, group = blockIdx.x / nsplit, split = blockIdx.x - group * nsplit;
    const int kh = group / a.ng, h0 = kh * a.kv_mul + (group - kh * a.ng) * QH;
    const int hn = min(min(h0 + QH, (kh + 1) * a.kv_mul), a.NH) - h0; /* heads of this group, 1 .. QH */
    const int c0 = split * a.keys, c1 = min(c0 + a.keys, a.S);
    const int row = lane / LPK, d4 = 4 * (lane % LPK);
    const float* kc = a.k + kh * HD + d4;
    const float* vc = a.v + kh * HD + d4;

    float4 kk[UN], vv[UN];
    auto fetch = [&](int base) { /* keys past the cache's S rows read row S - 1 and score -inf */
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const size_t off = (size_t)min(base + wave * T::WKEYS + u * T::KPI + row, a.S - 1) * a.KV;
            __builtin_memcpy(&kk[u], __builtin_assume_aligned(kc + off, 16), 16);
        }
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const size_t off = (size_t)min(base + wave * T::WKEYS + u * T::KPI + row, a.S - 1) * a.KV;
            __builtin_memcpy(&vv[u], __builtin_assume_aligned(vc + off, 16), 16);
        }
    };
    fetch(c0);
    float4 qv[QH];
#pragma unroll
    for (int i = 0; i < QH; i++) {
        const float* qh = a.q + (size_t)(h0 + min(i, hn - 1)) * HD + d4; /* 4-byte aligned */
        qv[i] = make_float4(qh[0], qh[1], qh[2], qh[3]);
    }
    float m[QH], l[QH];
    float4 acc[QH];
#pragma unroll
    for (int i = 0; i < QH; i++) {
        m[i] = -INFINITY;
        l[i] = 0.0f;
        acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int base = c0; base < c1; base += T::KEYS) {
        float s[QH][UN];
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const bool in = base + wave * T::WKEYS + u * T::KPI + row < c1;
#pragma unroll
            for (int i = 0; i < QH; i++) {
                const float d = fmaf(qv[i].x, kk[u].x, qv[i].y * kk[u].y) + fmaf(qv[i].z, kk[u].z, qv[i].w * kk[u].w);
                s[i][u] = in ? row_sum<LPK>(d) * a.scale : -INFINITY;
            }
        }
        float4 vt[UN];
#pragma unroll
        for (int u = 0; u < UN; u++) vt[u] = vv[u];
        if (base + T::KEYS < c1) fetch(base + T::KEYS);
#pragma unroll
        for (int i = 0; i < QH; i++) {
            float mt = s[i][0];
#pragma unroll
            for (int u = 1; u < UN; u++) mt = fmaxf(mt, s[i][u]);
#pragma unroll
            for (int o = LPK; o < 64; o <<= 1) mt = fmaxf(mt, __shfl_xor(mt, o));
            const float mn = fmaxf(m[i], mt);
            const float f = at_weight(m[i], mn);
            m[i] = mn;
            l[i] *= f;
            acc[i].x *= f;
            acc[i].y *= f;
            acc[i].z *= f;
            acc[i].w *= f;
#pragma unroll
            for (int u = 0; u < UN; u++) {
                const float p = at_weight(s[i][u], mn);
                l[i] += p;
                /* a masked key's row is another key's: it must not enter, whatever it holds */
                const bool in = base + wave * T::WKEYS + u * T::KPI + row < c1;
                acc[i].x = fmaf(p, in ? vt[u].x : 0.f, acc[i].x);
                acc[i].y = fmaf(p, in ? vt[u].y : 0.f, acc[i].y);
                acc[i].z = fmaf(p, in ? vt[u].z : 0.f, acc[i].z);
                acc[i].w = fmaf(p, in ? vt[u].w : 0.f, acc[i].w);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < QH; i++) {
#pragma unroll
        for (int o = LPK; o < 64; o <<= 1) {
            l[i] += __shfl_xor(l[i], o);
            acc[i].x += __shfl_xor(acc[i].x, o);
            acc[i].y += __shfl_xor(acc[i].y, o);
            acc[i].z += __shfl_xor(acc[i].z, o);
            acc[i].w += __shfl_xor(acc[i].w, o);
        }
        if (lane < LPK) *(float4*)&wacc[wave][i][d4] = acc[i];
        if (lane == 0) {
            wm[wave][i] = m[i];
            wl[wave][i] = l[i];
        }
    }
    __syncthreads();
    /* the workgroup's sum over its waves: thread (head i, dimension d), i * HD + d = t, t + AT_NT, ... */
    float* rec = a.rec + ((size_t)group * nsplit + split) * (QH * REC);
    for (int j = t; j < hn * HD; j += AT_NT) {
        const int i = j / HD, d = j - i * HD;
        float M = wm[0][i];
#pragma unroll
        for (int w = 1; w < AT_WAVES; w++) M = fmaxf(M, wm[w][i]);
        float L = 0.f, A = 0.f;
#pragma unroll
        for (int w = 0; w < AT_WAVES; w++) {
            const float f = at_weight(wm[w][i], M);
            L = fmaf(f, wl[w][i], L);
            A = fmaf(f, wacc[w][i][d], A);
        }
        if (nsplit == 1) {
            a.out[(size_t)(h0 + i) * HD + d] = A / L;
        } else {
            agent_store(&rec[i * REC + d], A);
            if (d == 0) {
                agent_store(&rec[i * REC + HD], M);
                agent_store(&rec[i * REC + HD + 1], L);
            }
        }
    }
    if (nsplit == 1) return;
    /* Records cross XCDs: they are written and read with agent-scope
     * accesses, which bypass the XCDs' own L2s, and each wave waits for its
     * stores before the barrier, so a workgroup is counted only after its
     * record has arrived.  (A fence would write back and invalidate a whole
     * L2 for these few hundred bytes.) */
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (t == 0) {
        unsigned int* done = &a.done[group * AT_DONE_STRIDE];
        const unsigned int n = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = n == (unsigned int)nsplit - 1u;
        if (last) __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return;
    const float* recs = a.rec + (size_t)group * nsplit * (QH * REC);
    /* wave i weighs head i's records: lane sp holds split sp */
    static_assert(QH <= AT_WAVES && AT_MAX_SPLIT <= 64, "a wave per head, a lane per split");
    if (wave < hn) {
        const bool in = lane < nsplit;
        const float* r = &recs[(size_t)min(lane, nsplit - 1) * (QH * REC) + wave * REC + HD];
        const float mi = in ? agent_load(r) : -INFINITY, li = in ? agent_load(r + 1) : 0.0f;
        const float f = at_weight(mi, wave_max(mi));
        rf[wave][lane] = f;
        const float L = wave_sum(f * li);
        if (lane == 0) rl[wave] = L;
    }
    __syncthreads();
    for (int j = t; j < hn * HD; j += AT_NT) {
        const int i = j / HD, d = j - i * HD;
        float A = 0.f;
        for (int b = 0; b < nsplit; b += 16) { /* 16 loads in flight; none past the records */
            float p[16];
#pragma unroll
            for (int e = 0; e < 16; e++)
                p[e] = b + e < nsplit ? agent_load(&recs[(size_t)(b + e) * (QH * REC) + i * REC + d]) : 0.0f;
#pragma unroll
            for (int e = 0; e < 16; e++) A = fmaf(b + e < nsplit ? rf[i][b + e] : 0.0f, p[e], A);
        }
        a.out[(size_t)(h0 + i) * HD + d] = A / rl[i];
    }
}

/* Up to two tiles of keys take one split (no records, no merge) and one query
 * head per workgroup: the scores of several heads one after another cost more
 * than what they share of so few rows.  us by kernel trace, workgroup per head
 * before the splits / shared heads / now, per head size and kv_mul: 64, 3: 16 keys
 * 5.0 / 4.3 / 3.2, 128 7.4 / 5.9 / 3.9; 128, 4: 65 8.9 / 10.2 / 5.4; 32, 4: 1 4.1 / 5.0 / 3.3;
 * 16, 4: 48 4.1 / 4.6 / 3.3; 256, 4: 48 13.4 / 15.0 / 5.7.  Three or four tiles of shared
 * heads in one split are faster too (64, 3, 256 keys 6.6 / 5.2), but the sums of a
 * workgroup get longer (error against 64 bits 1.41e-7 / 1.51e-7; 128, 4: 1.56e-7 /
 * 1.80e-7). */
constexpr int AT_ONE_TILES = 2;

/* Keys per split (*keys, whole tiles) and splits: one (AT_ONE_TILES), else as
 * many splits as there are tiles, up to AT_MAX_SPLIT and what the scratch
 * memory holds. */
template <int HD>
int at_split(int S, int groups, int qh, size_t scratch_bytes, int* keys) {
    const int tile = AtTile<HD>::KEYS, tiles = (S + tile - 1) / tile;
    size_t most = 1;
    if (tiles > AT_ONE_TILES && groups <= AT_MAX_GROUPS && scratch_bytes > AT_DONE_BYTES)
        most = (scratch_bytes - AT_DONE_BYTES) / ((size_t)groups * qh * (HD + 2) * 4);
    most = std::min<size_t>(std::max<size_t>(most, 1), AT_MAX_SPLIT);
    const int per = (tiles + (int)most - 1) / (int)most;
    *keys = per * tile;
    return (tiles + per - 1) / per;
}

template <int HD>
int at_launch(AtArgs a, int groups, int qh, const bmk_launch_t* l) {
    if (a.S <= AT_ONE_TILES * AtTile<HD>::KEYS) { /* one head per workgroup */
        qh = 1;
        a.ng = a.kv_mul;
        groups = a.NH;
    }
    a.nsplit = at_split<HD>(a.S, groups, qh, l->scratch_bytes, &a.keys);
    a.done = (unsigned int*)l->scratch;
    a.rec = a.nsplit > 1 ? (float*)((char*)l->scratch + AT_DONE_BYTES) : nullptr;
    const dim3 grid((unsigned)groups * a.nsplit), tb(AT_NT);
    if (qh == 1) hipLaunchKernelGGL((k_attn_decode<HD, 1>), grid, tb, 0, l->stream, a);
    else if (qh == 2) hipLaunchKernelGGL((k_attn_decode<HD, 2>), grid, tb, 0, l->stream, a);
    else if (qh == 3) hipLaunchKernelGGL((k_attn_decode<HD, 3>), grid, tb, 0, l->stream, a);
    else hipLaunchKernelGGL((k_attn_decode<HD, 4>), grid, tb, 0, l->stream, a);
    BMK_LAUNCH_CHECK();
    return 0;
}

} // namespace

/* attention_forward {q [NH][HD], kv cache, out [NH][HD],
 *                    params int{NH, HD, NKV, KV, S, kv_mul, layer, MS}, scale float} */
extern "C" int bmk_launch_attention(const bmk_launch_t* a) {
    BMK_NEED_BYTES(a, 3, 32, "params");
    BMK_NEED_BYTES(a, 4, 4, "scale");
    const int NH = bmk_pi(a, 3, 0), HD = bmk_pi(a, 3, 1), KV = bmk_pi(a, 3, 3), S = bmk_pi(a, 3, 4);
    const int kv_mul = bmk_pi(a, 3, 5), layer = bmk_pi(a, 3, 6), MS = bmk_pi(a, 3, 7);
    BMK_REQUIRE(NH > 0 && HD > 0 && HD <= 256 && 256 % HD == 0 && HD % 4 == 0 && kv_mul > 0 && layer >= 0 && MS > 0 &&
                    S >= 1 && S <= MS && ((NH - 1) / kv_mul + 1) * HD <= KV,
                "attention: bad params NH=%d HD=%d KV=%d S=%d kv_mul=%d layer=%d MS=%d", NH, HD, KV, S, kv_mul, layer,
                MS);
    BMK_NEED_BYTES(a, 0, (size_t)NH * HD * 4, "q");
    BMK_NEED_BYTES(a, 1, ((size_t)layer * 2 + 2) * MS * KV * 4, "kv cache");
    BMK_NEED_BYTES(a, 2, (size_t)NH * HD * 4, "out");
    BMK_REQUIRE(((uintptr_t)a->dev[1] & 15) == 0 && KV % 4 == 0, "attention: kv cache rows must be 16-byte aligned");
    AtArgs k;
    k.q = (const float*)a->dev[0];
    k.k = (const float*)a->dev[1] + (size_t)layer * 2 * MS * KV;
    k.v = k.k + (size_t)MS * KV;
    k.out = (float*)a->dev[2];
    k.NH = NH;
    k.KV = KV;
    k.S = S;
    k.scale = bmk_pf(a, 4, 0);
    /* a KV head's query heads in groups of qh <= 4; a kv_mul past NH serves the NH heads there are */
    k.kv_mul = std::min(kv_mul, NH);
    k.ng = (k.kv_mul + 3) / 4;
    const int qh = (k.kv_mul + k.ng - 1) / k.ng;
    k.ng = (k.kv_mul + qh - 1) / qh;
    const int groups = (NH - 1) / k.kv_mul * k.ng + ((NH - 1) % k.kv_mul) / qh + 1;
    switch (HD) {
    case 4: return at_launch<4>(k, groups, qh, a);
    case 8: return at_launch<8>(k, groups, qh, a);
    case 16: return at_launch<16>(k, groups, qh, a);
    case 32: return at_launch<32>(k, groups, qh, a);
    case 64: return at_launch<64>(k, groups, qh, a);
    case 128: return at_launch<128>(k, groups, qh, a);
    default: return at_launch<256>(k, groups, qh, a);
    }
}
