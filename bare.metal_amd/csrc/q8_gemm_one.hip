/* SPDX-License-Identifier: MPL-2.0
 *
 * q8_gemm_one.hip — one prefill GEMM over Q8_0 or Q4_0 rows (matmul_forward_q8 / _q4 with
 * 16 rows or more), on gfx950 bf16 MFMA:
 *   C[m][n] = sum_k bf16(A[m][k]) * bf16(q[n][k] * scale[n][k/32])   (fp32 accumulate)
 *
 * Operands and roundings as q8_gemm.hip's; a single projection has tens to
 * a few hundred tiles, so what bounds it is the chain of K steps of one
 * workgroup, not the matrix cores: each step waits for its loads, converts
 * them into LDS and meets a barrier.  So a step is wide (KS columns), eight
 * waves share it (KP of them along K, summed in LDS at the end), the tile is
 * small enough that every CU has one, and the loads run two steps ahead.
 */
#include "bmk.h"
#include "q8_common.h"
#include "q8_gemm.h"

namespace {

using bmk::QFmt;
using bmk::QF_Q4;
using bmk::QF_Q8;
using bmk::q4_code;
using bmk::q8_byte;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int G1_NT = 512;

struct G1Args {
    const float* A;
    const unsigned char* W;
    float* C;
    int M, N, K, tiles_n;
};

/* fp32 pair -> packed bf16 pair, round to nearest even (v_cvt_pk_bf16_f32) */
__device__ __forceinline__ unsigned int pk(float lo, float hi) {
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, bf16x2));
}

/* Keeps what is computed from a loaded value behind this point: hoisted to
 * the end of the previous step it would wait for loads just issued. */
template <class T>
__device__ __forceinline__ void pin(T& v) { asm volatile("" : "+v"(v)); }

/* TM x TN 32 x 32 tiles per workgroup, KP waves along K for each
 * (TM * TN * KP = 8 waves), K steps of KS columns. */
template <int QF, int TM, int TN, int KP, int KS>
__global__ __launch_bounds__(G1_NT) void k_gemm_one(G1Args a) {
    static_assert(TM * TN * KP == 8 && KS % (16 * KP) == 0, "eight waves, whole MFMAs");
    constexpr int BYTES = QFmt<QF>::BYTES;
    constexpr int LD = KS + 8;                                   /* LDS row in bf16; shifts rows by four banks */
    constexpr int AC = KS / 4, AP = 32 * TM * AC / G1_NT;        /* float4 chunks of an A row, chunks per thread */
    constexpr int WC = KS / 16, WP = 32 * TN * WC / G1_NT;       /* half blocks of a W row, per thread */
    static_assert(AP >= 1 && WP >= 1 && G1_NT % AC == 0 && G1_NT % WC == 0, "whole loader passes");
    constexpr int XF = 32 * TM * LD, BUF = 32 * (TM + TN) * LD;
    constexpr int LP = 33, PART = 8 * 32 * LP * 2;               /* the epilogue's partial tiles, in bf16 elements */
    __shared__ __attribute__((aligned(16))) unsigned short lds[2 * BUF > PART ? 2 * BUF : PART];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int wk = wave % KP, wt = wave / KP, wm = wt % TM, wn = wt / TM;
    const int r32 = lane & 31, h = lane >> 5;
    const int tm = blockIdx.x / a.tiles_n, tn = blockIdx.x - tm * a.tiles_n;
    const int m0 = tm * 32 * TM, n0 = tn * 32 * TN;
    const int nb = a.K / 32, nfull = a.K / KS;

    /* loaders: rows past M or N feed outputs that are not stored */
    const int ac = 4 * (t % AC), wb = (t % WC) >> 1, wh = t & 1;
    const float* ap[AP];
    const unsigned char* wp[WP];
#pragma unroll
    for (int p = 0; p < AP; p++) ap[p] = a.A + (size_t)min(m0 + t / AC + G1_NT / AC * p, a.M - 1) * a.K;
#pragma unroll
    for (int p = 0; p < WP; p++) wp[p] = a.W + (size_t)min(n0 + t / WC + G1_NT / WC * p, a.N - 1) * ((size_t)nb * BYTES);
    struct Stage {
        f32x4 x[AP];
        float s[WP];
        u32x4 q[WP]; /* 16 codes: int8, or nibbles in the first two dwords */
    };
    auto load = [&](int step, Stage& st) { /* past K: the row's last chunk, zeroed when the ragged step is stored */
        const int ka = min(step * KS + ac, a.K - 4), kb = min(step * (KS / 32) + wb, nb - 1);
#pragma unroll
        for (int p = 0; p < AP; p++) {
            f32x4 v;
            __builtin_memcpy(&v, __builtin_assume_aligned(ap[p] + ka, 4), 16);
            st.x[p] = v;
        }
#pragma unroll
        for (int p = 0; p < WP; p++) {
            const unsigned char* blk = wp[p] + (size_t)kb * BYTES;
            float s;
            __builtin_memcpy(&s, __builtin_assume_aligned(blk, 4), 4);
            st.s[p] = s;
            if (QF == QF_Q8) {
                u32x4 q;
                __builtin_memcpy(&q, __builtin_assume_aligned(blk + 4 + 16 * wh, 4), 16);
                st.q[p] = q;
            } else {
                u32x2 q;
                __builtin_memcpy(&q, __builtin_assume_aligned(blk + 4 + 8 * wh, 4), 8);
                st.q[p] = u32x4{q.x, q.y, 0u, 0u};
            }
        }
    };
    auto store = [&](int buf, const Stage& st, bool ina, bool inw) { /* ina, inw: this thread's chunks lie inside K */
        unsigned short* As = lds + buf * BUF;
        unsigned short* Ws = As + XF;
#pragma unroll
        for (int p = 0; p < AP; p++) {
            f32x4 x = st.x[p];
            pin(x);
            x = ina ? x : f32x4{0.f, 0.f, 0.f, 0.f};
            const u32x2 u = {pk(x.x, x.y), pk(x.z, x.w)};
            *(u32x2*)&As[(t / AC + G1_NT / AC * p) * LD + ac] = u;
        }
#pragma unroll
        for (int p = 0; p < WP; p++) {
            unsigned short* d = &Ws[(t / WC + G1_NT / WC * p) * LD + 32 * wb + 16 * wh];
            u32x4 q = st.q[p];
            float s = st.s[p];
            pin(q);
            pin(s);
            s = inw ? s : 0.0f;
            u32x4 lo, hi;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (QF == QF_Q8) {
                    const unsigned int w0 = q[j >> 1], w1 = q[2 + (j >> 1)];
                    lo[j] = pk(q8_byte(w0, 2 * (j & 1)) * s, q8_byte(w0, 2 * (j & 1) + 1) * s);
                    hi[j] = pk(q8_byte(w1, 2 * (j & 1)) * s, q8_byte(w1, 2 * (j & 1) + 1) * s);
                } else {
                    lo[j] = pk(q4_code(q.x, 2 * j) * s, q4_code(q.x, 2 * j + 1) * s);
                    hi[j] = pk(q4_code(q.y, 2 * j) * s, q4_code(q.y, 2 * j + 1) * s);
                }
            }
            *(u32x4*)d = lo;
            *(u32x4*)(d + 8) = hi;
        }
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    constexpr int KW = KS / KP; /* a wave's columns of a step */
    struct Frags {
        bf16x8 a[KW / 16], w[KW / 16];
    };
    auto frags = [&](int buf, Frags& f) {
        const unsigned short* As = lds + buf * BUF + (32 * wm + r32) * LD + KW * wk + 8 * h;
        const unsigned short* Ws = lds + buf * BUF + XF + (32 * wn + r32) * LD + KW * wk + 8 * h;
#pragma unroll
        for (int k = 0; k < KW / 16; k++) {
            f.a[k] = *(const bf16x8*)(As + 16 * k);
            f.w[k] = *(const bf16x8*)(Ws + 16 * k);
        }
    };
    auto mfma = [&](const Frags& f) {
#pragma unroll
        for (int k = 0; k < KW / 16; k++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[k], f.w[k], acc, 0, 0, 0);
    };
    auto mfma_step = [&](int buf) {
        Frags f;
        frags(buf, f);
        mfma(f);
    };
    /* Full steps: step s computes from buffer s & 1 while the loads of step
     * s + 2 are in flight (past the last one they repeat it and feed nothing).
     * A step's fragments are read before the next step is converted and
     * multiplied after it, so that the conversions, which are most of a step,
     * cover the reads: 333 x 2560 -> 960 14.0 -> 12.8 us, 960 -> 2560 9.8 -> 9.4.
     * The ragged step's loads are issued up front and wait in registers of
     * their own: a select or a branch on the loop's stages makes the compiler
     * wait for every load in flight. */
    const bool ragged = a.K % KS != 0;
    Stage s0, s1, sr;
    if (nfull > 0) {
        load(0, s0);
        load(min(1, nfull - 1), s1);
    }
    if (ragged) load(nfull, sr);
    if (nfull > 0) {
        store(0, s0, true, true);
        __syncthreads();
        int step = 0;
        for (; step + 2 <= nfull; step += 2) {
            load(min(step + 2, nfull - 1), s0);
            Frags f0;
            frags(0, f0);
            __builtin_amdgcn_sched_barrier(0);
            store(1, s1, true, true);
            __builtin_amdgcn_sched_barrier(0);
            mfma(f0);
            __syncthreads();
            load(min(step + 3, nfull - 1), s1);
            Frags f1;
            frags(1, f1);
            __builtin_amdgcn_sched_barrier(0);
            store(0, s0, true, true);
            __builtin_amdgcn_sched_barrier(0);
            mfma(f1);
            __syncthreads();
        }
        if (step < nfull) mfma_step(0); /* odd step count: the last step sits in buffer 0 */
    }
    if (ragged) { /* buffer nfull & 1 is free: a barrier followed its last reader */
        store(nfull & 1, sr, nfull * KS + ac < a.K, nfull * (KS / 32) + wb < nb);
        __syncthreads();
        mfma_step(nfull & 1);
    }
    __syncthreads();
    /* the KP parts of each tile, summed in wave order (every wave is past its
     * reads of LDS); register r of a tile: row 8 (r / 4) + 4 (lane / 32) + r % 4,
     * column lane % 32 */
    float* parts = (float*)lds;
#pragma unroll
    for (int r = 0; r < 16; r++) parts[(wave * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * LP + r32] = acc[r];
    __syncthreads();
    const int row = t >> 5, col = t & 31;
#pragma unroll
    for (int i = 0; i < TM * TN * 2; i++) { /* 16 rows of tile i / 2 */
        const int tile = i >> 1, rr = 16 * (i & 1) + row;
        const int m = m0 + 32 * (tile % TM) + rr, n = n0 + 32 * (tile / TM) + col;
        if (m >= a.M || n >= a.N) continue;
        const float* src = parts + (tile * KP * 32 + rr) * LP + col;
        float v = src[0];
#pragma unroll
        for (int k = 1; k < KP; k++) v += src[k * 32 * LP];
        a.C[(size_t)m * a.N + n] = v;
    }
}

template <int QF, int TM, int TN, int KP, int KS>
void g1_go(G1Args a, hipStream_t s) {
    a.tiles_n = (a.N + 32 * TN - 1) / (32 * TN);
    const unsigned tiles_m = (a.M + 32 * TM - 1) / (32 * TM);
    hipLaunchKernelGGL((k_gemm_one<QF, TM, TN, KP, KS>), dim3(tiles_m * a.tiles_n), dim3(G1_NT), 0, s, a);
}

/* 1: launched; 0: more tiles than CUs even at 64 x 128; -1: the launch failed */
template <int QF>
int g1_pick(const G1Args& a, hipStream_t s) {
    constexpr long CUS = 256;
    auto tiles = [&](long tm, long tn) { return ((a.M + tm - 1) / tm) * ((a.N + tn - 1) / tn); };
    if (tiles(32, 32) <= CUS) g1_go<QF, 1, 1, 8, 256>(a, s);
    else if (tiles(32, 64) <= CUS) g1_go<QF, 1, 2, 4, 128>(a, s);
    else if (tiles(64, 64) <= CUS) g1_go<QF, 2, 2, 2, 128>(a, s);
    else if (tiles(64, 128) <= CUS) g1_go<QF, 2, 4, 1, 64>(a, s);
    else return 0;
    BMK_LAUNCH_CHECK();
    return 1;
}

} // namespace

/* The shape is the smallest tile that one workgroup per CU covers; past the
 * largest the launch belongs to the 128 x 128 kernel, which dequantises each
 * weight for more rows.  GPU time per launch, back to back, in us (Q8_0; tiles of
 * 32 x 32 / 32 x 64 / 64 x 64 / 64 x 128 / 128 x 128, tile counts in brackets):
 *   64 x 960 -> 2560:    5.4 [160]   6.8 [80]    8.3 [40]   10.9 [20]   17.9
 *   128 x 960 -> 2560:   7.9 [320]   7.1 [160]   8.5 [80]   11.2 [40]   16.7
 *   333 x 960 -> 2560:  13.8 [880]  10.9 [440]   9.7 [240]  12.0 [120]  18.4
 *   512 x 960 -> 2560:  17.4        15.6 [640]  17.4 [320]  12.7 [160]  18.1
 *   1024 x 960 -> 2560: 32.8        25.7        25.8 [640]  19.7 [320]  19.3 [160]
 *   64 x 2560 -> 960:    9.0 [60]   12.6        16.3        24.2        40.2
 *   333 x 2560 -> 960:  14.9 [330]  13.8 [165]  17.6 [90]   24.6        41.4
 *   2048 x 2560 -> 960: 58.0        46.0        39.7 [480]  32.9 [256]  44.6
 *   512 x 1536 -> 576:  11.2 [288]   9.7 [144]  12.1        16.4        26.8
 *   1024 x 576 -> 1536: 20.2        13.3 [768]  15.2 [384]   9.7 [192]  12.6
 * 32 x 64 with steps of 256 instead of 128: 6.9, 7.1, 13.7, 20.0, 32.9, 12.7, 14.2.
 * (Taken before the fragments were read ahead, which took 2-8% off each.) */
extern "C" int gm_launch_one(const float* A, const unsigned char* W, float* C, int M, int N, int K, int qf,
                             hipStream_t s) {
    const G1Args a = {A, W, C, M, N, K, 0};
    if (qf == QF_Q4) return g1_pick<QF_Q4>(a, s);
    return g1_pick<QF_Q8>(a, s);
}
