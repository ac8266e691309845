/* SPDX-License-Identifier: MPL-2.0
 *
 * rows_gemm.hip — the plain matmul over unquantized rows for several input rows:
 *   out[b][r] = bias[r] + sum_k x[b][k] * w[r][k],  w fp32, bf16 or fp16 (widened exactly), fp32 products and sums.
 * Served names: matmul_forward_{naive,tiled,fp32_tiled,bf16*,fp16*} with several rows (decode.hip's launcher).
 *
 * The products run on v_mfma_f32_32x32x2_f32 (fp32 operands, so infinities,
 * NaN and the operands' 24 bits are the plain sum's).  What bounds it: the
 * matrix pipe's fp32 rate (157 TFLOP/s, 64 cycles an instruction) once the
 * operands come in whole lines, so both go through LDS: a workgroup loads
 * rows of a K step with full-line loads two steps ahead, widens the weights
 * while storing them, and its waves read fragments of four k at once
 * (conflict-free: rows are padded by four floats).
 * Two tile shapes (rg_launch):
 *   32 x 32, the four waves taking a quarter of each 128-wide K step, summed
 *   in LDS at the end: the most workgroups, for launches that fit one per CU,
 *   and for up to 32 rows, which a 64-row tile would leave half empty (8 x 960 ->
 *   49152 68.5 / 41.3 us, 16 x 2560 -> 8192 no different);
 *   64 x 32, two waves along the rows and two along K: a third less operand
 *   traffic per product where the CUs would take several workgroups each.
 * Measured, C = 960, bf16 rows, 32 x 32 / 64 x 32 (us, back to back, one
 * partial sum per wave in both): 64 x 2560 9.3 / 13.6, 100 x 2560 15.8 / 14.1,
 * 333 x 2560 29.3 / 24.9, 512 x 2560 37.1 / 36.3, 200 x 2560 22.7 / 23.8; C = 2560:
 * 333 x 960 33.4 / 32.8, 200 x 960 (210 tiles) 19.3 / 31.6.  64 x 64 over whole K
 * steps was slower than one of the two everywhere but at 333 x 2560 (24.0).
 * Against the LM-head kernel, whose workgroups apply their rows to each input
 * row in turn: 64 x 2560 190 -> 9.9 us, 512 x 2560 1560 -> 37 us.
 */
#include "bmk.h"
#include "rows_gemm.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int RG_NT = 256;
/* Partial sums a wave keeps in turn, and K steps after which the two-wave
 * form folds them into one: chains of about C / 64 roundings (32 x 32) and of
 * 16 (64 x 32), so the error against 64 bits is no larger than that of the
 * LM-head kernel's sums (normwise, C 960 / 2560: 1.2e-7 / 1.7e-7; with one
 * partial sum 2.8e-7, with four 1.5e-7 / 2.4e-7; eight cost 0.4 us). */
constexpr int ACC = 8, FOLD = 8;
/* a launch of more rows than a tile's and more 32 x 32 tiles than this (one per CU) takes 64 x 32 ones */
constexpr long RG_CU_TILES = 256;

struct RgArgs {
    const float* x;
    const void* w;
    const float* bias;
    float* out;
    int BT, C, OC;
};

/* 16 bytes from a 4-byte aligned address */
__device__ __forceinline__ f32x4 load16(const void* p) {
    f32x4 v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 4), 16);
    return v;
}

/* four weights from 4 (fp32) or 2 (16-bit) dwords */
template <int WF>
__device__ __forceinline__ f32x4 widen4(float f0, float f1) {
    const unsigned int u0 = __float_as_uint(f0), u1 = __float_as_uint(f1);
    f32x4 r;
    if (WF == RG_BF16) {
        r.x = __uint_as_float(u0 << 16);
        r.y = __uint_as_float(u0 & 0xffff0000u);
        r.z = __uint_as_float(u1 << 16);
        r.w = __uint_as_float(u1 & 0xffff0000u);
    } else {
        r.x = (float)__builtin_bit_cast(_Float16, (unsigned short)(u0 & 0xffffu));
        r.y = (float)__builtin_bit_cast(_Float16, (unsigned short)(u0 >> 16));
        r.z = (float)__builtin_bit_cast(_Float16, (unsigned short)(u1 & 0xffffu));
        r.w = (float)__builtin_bit_cast(_Float16, (unsigned short)(u1 >> 16));
    }
    return r;
}

/* TM 32 x 32 tiles per workgroup, KP waves along K for each (TM * KP = 4),
 * K steps of 32 * KP; C a multiple of 32. */
template <int WF, int TM, int KP>
__global__ __launch_bounds__(RG_NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_rows_gemm(RgArgs a) {
    static_assert(TM * KP == 4, "four waves");
    constexpr int KS = 32 * KP, LD = KS + 4;           /* LDS row in floats */
    constexpr int XC = KS / 4, XP = 32 * TM * XC / RG_NT; /* float4 chunks of an x row, chunks per thread */
    constexpr int WE = WF == RG_F32 ? 4 : 8;           /* weights per 16-byte chunk */
    constexpr int WC = KS / WE, WP = 32 * WC / RG_NT;
    constexpr int XF = 32 * TM * LD, BUF = 32 * (TM + 1) * LD;
    __shared__ __attribute__((aligned(16))) float lds[2 * BUF];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int wk = wave % KP, wm = wave / KP; /* wave = tile * KP + K part */
    const int r32 = lane & 31, h = lane >> 5;
    const int m0 = blockIdx.x * 32 * TM, n0 = blockIdx.y * 32;
    const int nstep = (a.C + KS - 1) / KS;

    /* loaders: rows past BT or OC and chunks past C read valid memory that feeds nothing stored */
    const float* xp[XP];
    const unsigned char* wp[WP];
    constexpr int WSZ = WF == RG_F32 ? 4 : 2;
    const int xc = 4 * (t % XC), wc = WE * (t % WC);
#pragma unroll
    for (int p = 0; p < XP; p++) xp[p] = a.x + (size_t)min(m0 + t / XC + RG_NT / XC * p, a.BT - 1) * a.C;
#pragma unroll
    for (int p = 0; p < WP; p++)
        wp[p] = (const unsigned char*)a.w + (size_t)min(n0 + t / WC + RG_NT / WC * p, a.OC - 1) * a.C * WSZ;
    struct Stage {
        f32x4 x[XP];
        f32x4 w[WP];
    };
    auto load = [&](int step, Stage& s) {
        const int kx = min(step * KS + xc, a.C - 4), kw = min(step * KS + wc, a.C - WE);
#pragma unroll
        for (int p = 0; p < XP; p++) s.x[p] = load16(xp[p] + kx);
#pragma unroll
        for (int p = 0; p < WP; p++) s.w[p] = load16(wp[p] + (size_t)kw * WSZ);
    };
    auto store = [&](int buf, const Stage& s) {
        float* xs = lds + buf * BUF;
        float* ws = xs + XF;
#pragma unroll
        for (int p = 0; p < XP; p++) *(f32x4*)&xs[(t / XC + RG_NT / XC * p) * LD + xc] = s.x[p];
#pragma unroll
        for (int p = 0; p < WP; p++) {
            float* d = &ws[(t / WC + RG_NT / WC * p) * LD + wc];
            if (WF == RG_F32) {
                *(f32x4*)d = s.w[p];
            } else {
                *(f32x4*)d = widen4<WF>(s.w[p].x, s.w[p].y);
                *(f32x4*)(d + 4) = widen4<WF>(s.w[p].z, s.w[p].w);
            }
        }
    };
    /* the output column of this thread in the epilogue, and its bias (nothing to add is -0: v + -0 is v for every v) */
    const int n = n0 + (t & 31);
    const float bv = a.bias && n < a.OC ? a.bias[n] : -0.0f;
    f32x16 acc[ACC], tot;
#pragma unroll
    for (int i = 0; i < ACC; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = tot[r] = 0.0f;
    auto fold = [&]() { return ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7])); };
    static_assert(ACC == 8 && FOLD % 2 == 0, "fold adds eight, the loop takes two steps");
    auto mfma_step = [&](int buf, int step) {
        if (step * KS + 32 * wk >= a.C) return; /* the last step may not reach this wave's part (wave-uniform) */
        const float* xs = lds + buf * BUF + (32 * wm + r32) * LD + 32 * wk + 4 * h;
        const float* ws = lds + buf * BUF + XF + r32 * LD + 32 * wk + 4 * h;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const f32x4 av = *(const f32x4*)(xs + 8 * j), bv = *(const f32x4*)(ws + 8 * j);
#pragma unroll
            for (int e = 0; e < 4; e++)
                acc[(4 * j + e) % ACC] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[e], bv[e], acc[(4 * j + e) % ACC], 0, 0, 0);
        }
    };
    /* step s computes from buffer s & 1 while the loads of step s + 2 are in
     * flight; past the last step they repeat it and feed nothing */
    Stage s0, s1;
    load(0, s0);
    load(min(1, nstep - 1), s1);
    store(0, s0);
    __syncthreads();
    for (int step = 0; step < nstep; step += 2) {
        if (KP == 2 && step && step % FOLD == 0) {
            tot += fold();
#pragma unroll
            for (int i = 0; i < ACC; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;
        }
        load(min(step + 2, nstep - 1), s0);
        __builtin_amdgcn_sched_barrier(0);
        mfma_step(0, step);
        __builtin_amdgcn_sched_barrier(0);
        store(1, s1);
        __syncthreads();
        if (step + 1 >= nstep) break;
        load(min(step + 3, nstep - 1), s1);
        __builtin_amdgcn_sched_barrier(0);
        mfma_step(1, step + 1);
        __builtin_amdgcn_sched_barrier(0);
        store(0, s0);
        __syncthreads();
    }
    /* the K parts of each tile, summed in wave order (every wave is past its
     * reads of LDS); register r of a tile: row 8 (r / 4) + 4 (lane / 32) + r % 4,
     * column lane % 32 */
    constexpr int LP = 33;
    float* part = lds + wave * 32 * LP;
    tot += fold();
#pragma unroll
    for (int r = 0; r < 16; r++) part[(8 * (r >> 2) + 4 * h + (r & 3)) * LP + r32] = tot[r];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 4 * TM; p++) {
        const int row = t / 32 + 8 * p, m = m0 + row;
        if (m >= a.BT || n >= a.OC) continue;
        const float* src = lds + ((row >> 5) * KP * 32 + (row & 31)) * LP + (t & 31);
        float v = src[0] + src[32 * LP];
        if (KP == 4) v += src[2 * 32 * LP] + src[3 * 32 * LP];
        a.out[(size_t)m * a.OC + n] = bv + v;
    }
}

template <int WF>
void rg_launch(const RgArgs& a, hipStream_t s) {
    const unsigned tn = (a.OC + 31) / 32;
    if (a.BT > 32 && (long)((a.BT + 31) / 32) * tn > RG_CU_TILES)
        hipLaunchKernelGGL((k_rows_gemm<WF, 2, 2>), dim3((a.BT + 63) / 64, tn), dim3(RG_NT), 0, s, a);
    else
        hipLaunchKernelGGL((k_rows_gemm<WF, 1, 4>), dim3((a.BT + 31) / 32, tn), dim3(RG_NT), 0, s, a);
}

} // namespace

/* A few rows stay with the LM-head kernel, which reads its weights once and
 * applies them to each row in turn, where that takes less than a 32-row tile.
 * Its cost grows with the rows and little with OC while the CUs last; here it is
 * the chain over C, and past one tile per CU the tiles' count.  Both sides in
 * us (head kernel / this one, kernel trace, bf16 rows):
 *   up to one tile per CU   C = 960        1536         2560         4096         8192
 *     2 rows                9.3 / 8.5      11.2 / 12.2  13.3 / 18.6  17.0 / 27.6  26.4 / 53.8
 *     3 rows                12.2 / 8.8     15.3 / 12.0  18.2 / 18.6  23.6 / 27.6  37.1 / 53.2
 *     4 rows                15.4 / 8.5     19.0 / 12.0  23.0 / 18.6  30.3 / 27.6  47.9 / 53.2
 *     5 rows                18.3 / 8.9     22.8 / 12.2  27.8 / 18.5  37.1 / 27.6  59.3 / 53.4
 *   more                    960 -> 16384   960 -> 49152 2048 -> 32000  4096 -> 16384
 *     2 rows                10.3 / 15.8    34.3 / 44.1  60.4 / 55.8    76.0 / 55.2
 *     3 rows                13.0 / 15.6    42.8 / 43.7  79.2 / 55.0    102.8 / 54.5
 *     4 rows                16.2 / 15.6    51.7 / 43.0  98.2 / 54.3    129.5 / 54.5
 * fp32 rows differ at three: 2560 -> 960 23.5 / 20.2, 4096 -> 40 34.1 / 29.8, 960 -> 49152 42.2 / 45.6, 8192 -> 2048
 * 34.6 / 59.0 (five rows 57.8 / 59.5). */
extern "C" int rows_gemm_ok(int BT, int C, int OC, int wf) {
    if (BT < 2 || C % 32 != 0 || OC > 65535L * 32) return 0;
    if ((OC + 31) / 32 > RG_CU_TILES) return BT >= 4 || C >= 2048;
    const int most = BT == 2 ? 1024 : BT == 3 ? (wf == RG_F32 ? 4096 : 2560) : BT == 4 ? 4096 : C;
    return C <= most;
}

extern "C" int rows_gemm_launch(const float* x, const void* w, int wf, const float* bias, float* out, int BT, int C,
                                int OC, hipStream_t s) {
    /* the loaders take 16 bytes from 4-byte aligned addresses, 16-bit weights too */
    BMK_REQUIRE(BT > 0 && OC > 0 && C > 0 && C % 32 == 0 && OC <= 65535L * 32, "rows gemm: %d x %d -> %d", BT, C, OC);
    BMK_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 3) == 0, "rows gemm: operands must be 4-byte aligned");
    const RgArgs a = {x, w, bias, out, BT, C, OC};
    if (wf == RG_F32) rg_launch<RG_F32>(a, s);
    else if (wf == RG_BF16) rg_launch<RG_BF16>(a, s);
    else rg_launch<RG_F16>(a, s);
    BMK_LAUNCH_CHECK();
    return 0;
}
