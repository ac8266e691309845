/* SPDX-License-Identifier: MPL-2.0
 *
 * persist_cpu.cpp — the persistent decode step's kernel run on the CPU, one fiber per lane, to show that its result
 * does not depend on the order in which waves run (test_persist_order.py builds it around decode_persist.hip).
 *
 * Lanes switch only where the hardware would make a wave wait: at a cross-lane operation, at a workgroup barrier and
 * in a poll of exchanged values.  A run holds one wave of one workgroup back as long as anything else in the grid can
 * go on, so whatever that wave reads without a barrier in between is overwritten before it reads it.
 *
 * usage: persist_cpu NB NH NKV pos first step: holds back waves first, first + step, ... of the grid, one a run;
 * prints "runs N differ M", exit status 0 (nothing differs), 1, or 2 (a run stuck)
 */
#include <math.h>
#include <setjmp.h>
#include <stdarg.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <map>
#include <memory>
#include <string>
#include <vector>

/* ---------------- the part of HIP that the kernel uses */
using std::max;
using std::min;
#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
typedef void* hipStream_t;
typedef int hipError_t;
enum { hipSuccess = 0 };
static hipError_t hipGetLastError() { return hipSuccess; }
static const char* hipGetErrorString(hipError_t) { return ""; }
struct uint4 { unsigned int x, y, z, w; };
struct alignas(16) float4 { float x, y, z, w; };
static uint4 make_uint4(unsigned x, unsigned y, unsigned z, unsigned w) { return {x, y, z, w}; }
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
static unsigned __float_as_uint(float f) { return __builtin_bit_cast(unsigned, f); }
static float __uint_as_float(unsigned u) { return __builtin_bit_cast(float, u); }
extern "C" void bmk_log(const char*, const char*, int, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vfprintf(stderr, fmt, ap);
    va_end(ap);
}

/* ---------------- lanes, waves, workgroups */
namespace emu {

constexpr int NL = 64, NWAVE = 4;
constexpr size_t STACK = 32768 + 5 * 64; /* not a power of two, for the caches */

struct Lane {
    jmp_buf at;
    bool started = false, done = false;
    unsigned barrier_gen = 0, seen = 0;
    enum { RUN, BARRIER, STORE } wait = RUN;
};
struct Wave {
    Lane lane[NL];
    uint64_t slot[2][NL];
    unsigned stores[2]; /* emu::stores when the last lane arrived */
    unsigned gen = 0;
    int arrived = 0;
};
struct Group {
    unsigned block;
    Wave wave[NWAVE];
    char* stacks; /* one of stack_pool's, kept from run to run */
    std::map<std::string, std::vector<char>> lds;
    unsigned barrier_gen = 0;
    int arrived = 0, live = NL * NWAVE;
};

static std::vector<std::unique_ptr<char[]>> stack_pool;
static std::function<void()> body;
static Group* grp;
static Wave* wave;
static Lane* lane;
static int thread;
static jmp_buf scheduler;
static unsigned stores; /* counts stores of exchanged values: what a poll waits for */

static void yield() {
    if (!_setjmp(lane->at)) _longjmp(scheduler, 1);
}
static void open_barrier(Group* g) {
    if (g->arrived < g->live || !g->live) return;
    g->arrived = 0;
    g->barrier_gen++;
}
static void entry() {
    body();
    lane->done = true;
    grp->live--;
    open_barrier(grp); /* a lane that has ended is not waited for */
    _longjmp(scheduler, 1);
}
/* every lane's value, once all lanes of the wave have arrived */
static const uint64_t* all_lanes(uint64_t v) {
    Wave& w = *wave;
    const unsigned g = w.gen;
    w.slot[g & 1][thread % NL] = v;
    if (++w.arrived == NL) {
        w.arrived = 0;
        w.stores[g & 1] = stores;
        w.gen++;
    } else {
        while (w.gen == g) yield();
    }
    return w.slot[g & 1];
}
template <class T>
static T from_lane(T v, int src) {
    uint64_t u = 0;
    memcpy(&u, &v, sizeof v);
    T r;
    memcpy(&r, &all_lanes(u)[src], sizeof r);
    return r;
}
static void barrier() {
    lane->barrier_gen = grp->barrier_gen;
    lane->wait = Lane::BARRIER;
    grp->arrived++;
    open_barrier(grp);
    while (lane->barrier_gen == grp->barrier_gen) yield();
    lane->wait = Lane::RUN;
}
/* a wave's failed poll: again at once if a lane's loads are older than a store, else after the next store */
static unsigned long long poll_pause() {
    const unsigned g = wave->gen & 1;
    const uint64_t* s = all_lanes(lane->seen);
    const unsigned now = wave->stores[g];
    if (std::all_of(s, s + NL, [=](uint64_t v) { return v == now; })) {
        lane->wait = Lane::STORE;
        lane->seen = now;
        while (lane->seen == stores) yield();
        lane->wait = Lane::RUN;
    }
    lane->seen = stores;
    return 0;
}
static void* lds(const char* name, size_t n) {
    std::vector<char>& v = grp->lds[name];
    if (v.empty()) v.assign(n, (char)0xff); /* NaN */
    return v.data();
}

static void resume(Group* g, int w, int l) {
    grp = g;
    wave = &g->wave[w];
    lane = &wave->lane[l];
    thread = w * NL + l;
    if (_setjmp(scheduler)) return;
    if (lane->started) _longjmp(lane->at, 1);
    lane->started = true;
    ucontext_t c;
    getcontext(&c);
    c.uc_stack.ss_sp = g->stacks + STACK * thread;
    c.uc_stack.ss_size = STACK;
    c.uc_link = nullptr;
    makecontext(&c, entry, 0);
    setcontext(&c);
}
/* each lane of the wave that can go on, to its next stop */
static bool pass(Group* g, int w) {
    bool any = false;
    for (int l = 0; l < NL; l++) {
        Lane& a = g->wave[w].lane[l];
        if (a.done || (a.wait == Lane::BARRIER && a.barrier_gen == g->barrier_gen) ||
            (a.wait == Lane::STORE && a.seen == stores))
            continue;
        const unsigned gen = g->wave[w].gen;
        const int arrived = g->wave[w].arrived;
        const bool was = a.started;
        resume(g, w, l);
        /* a lane that is still waiting for its wave has not moved */
        any = any || !was || a.done || a.wait != Lane::RUN || gen != g->wave[w].gen || arrived != g->wave[w].arrived;
    }
    return any;
}

static int late_group = -1, late_wave; /* the wave held back (late_group < 0: none) */
static bool stuck;

static void launch(dim3 grid, std::function<void()> f) {
    body = f;
    std::vector<std::unique_ptr<Group>> gs;
    for (unsigned b = 0; b < grid.x; b++) {
        std::unique_ptr<Group> g(new Group);
        g->block = b;
        if (stack_pool.size() <= gs.size()) stack_pool.emplace_back(new char[STACK * NL * NWAVE]);
        g->stacks = stack_pool[gs.size()].get();
        pass(g.get(), NWAVE - 1); /* workgroups without work end at once */
        if (g->wave[NWAVE - 1].lane[0].done) continue;
        gs.push_back(std::move(g));
    }
    for (;;) {
        bool any = false, live = false;
        for (size_t g = 0; g < gs.size(); g++)
            for (int w = 0; w < NWAVE; w++)
                if (!((int)g == late_group && w == late_wave))
                    while (pass(gs[g].get(), w)) any = true;
        if (any) continue;
        if (late_group >= 0 && pass(gs[late_group].get(), late_wave)) continue;
        for (auto& g : gs) live = live || g->live;
        stuck = live;
        return;
    }
}

} // namespace emu

struct EmuIdx {
    struct X {
        operator unsigned() const { return emu::thread; }
    } x;
};
struct EmuBlock {
    struct X {
        operator unsigned() const { return emu::grp->block; }
    } x;
};
static EmuIdx threadIdx;
static EmuBlock blockIdx;

#define __HIP_MEMORY_SCOPE_WAVEFRONT 0
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, order, scope) (*(p))
#define __hip_atomic_store(p, v, order, scope) (*(p) = (v), (void)emu::stores++)
static unsigned atomicOr(unsigned* p, unsigned v) { const unsigned o = *p; *p |= v; return o; }
static unsigned atomicExch(unsigned* p, unsigned v) { const unsigned o = *p; *p = v; return o; }
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_sched_barrier(m) ((void)0)
#define __builtin_amdgcn_s_setprio(p) ((void)0)
#define __builtin_amdgcn_s_getreg(r) 0
#define __builtin_amdgcn_cvt_off_f32_i4(v) ((float)((int)((unsigned)(v) << 28) >> 28) / 16.0f)
#define __builtin_amdgcn_s_barrier() emu::barrier()
#define __builtin_amdgcn_wave_barrier() ((void)emu::all_lanes(0))
#define __builtin_amdgcn_s_memrealtime() emu::poll_pause()
#define __builtin_amdgcn_readlane(v, l) emu::from_lane(v, l)
#define __builtin_amdgcn_readfirstlane(v) emu::from_lane(v, 0)
static float __shfl_xor(float v, int m, int = 64) { return emu::from_lane(v, (emu::thread % 64) ^ m); }
static int __builtin_amdgcn_update_dpp(int, int v, int ctrl, int, int, bool) {
    const int l = emu::thread % 64;
    const int src = ctrl == 0xB1 ? l ^ 1 : ctrl == 0x4E ? l ^ 2 : ctrl == 0x141 ? l ^ 7 : ctrl == 0x140 ? l ^ 15 : -1;
    if (src < 0) abort();
    return emu::from_lane(v, src);
}
struct EmuPair {
    unsigned v[2];
    unsigned operator[](int i) const { return v[i]; }
};
static EmuPair __builtin_amdgcn_permlane32_swap(unsigned a, unsigned b, bool, bool) {
    const int l = emu::thread % 64;
    const uint64_t* s = emu::all_lanes(a | (uint64_t)b << 32);
    const unsigned lo_a = (unsigned)s[l & 31], hi_a = (unsigned)s[(l & 31) + 32];
    const unsigned lo_b = (unsigned)(s[l & 31] >> 32), hi_b = (unsigned)(s[(l & 31) + 32] >> 32);
    return {{l < 32 ? lo_a : lo_b, l < 32 ? hi_a : hi_b}}; /* a's upper half and b's lower half swapped */
}
static bool __all(bool p) {
    const uint64_t* s = emu::all_lanes(p);
    return std::all_of(s, s + 64, [](uint64_t v) { return v != 0; });
}
#define hipLaunchKernelGGL(k, grid, block, sh, stream, args) emu::launch(grid, [=] { k(args); })

/* the kernel, its LDS declarations turned into calls of emu::lds and its empty asm statements taken out */
#include "decode_persist.cpp"

/* ---------------- one step of a small model under every order */
int main(int argc, char** argv) {
    if (argc != 7) return 2;
    const int first = atoi(argv[5]), step = atoi(argv[6]);
    const int NB = atoi(argv[1]), NH = atoi(argv[2]), NKV = atoi(argv[3]), pos = atoi(argv[4]);
    const int D = 64, H = 64, L = 2, MS = pos + 8;
    const int QD = NH * 64, KV = NKV * 64;
    uint64_t rng = 88172645463325252ull;
    auto uni = [&] { /* xorshift64, uniform in [-1, 1) */
        rng ^= rng << 13;
        rng ^= rng >> 7;
        rng ^= rng << 17;
        return (float)((int64_t)rng >> 40) / 8388608.0f;
    };
    DecPersist a;
    memset(&a, 0, sizeof a);
    const size_t rows[7] = {(size_t)QD, (size_t)KV, (size_t)KV, (size_t)D, (size_t)H, (size_t)H, (size_t)D};
    const size_t cols[7] = {(size_t)D, (size_t)D, (size_t)D, (size_t)QD, (size_t)D, (size_t)D, (size_t)H};
    size_t bytes = 0;
    for (int m = 0; m < 7; m++) {
        a.off[m] = bytes;
        bytes += rows[m] * cols[m] / 32 * 36;
    }
    a.layer_bytes = bytes;
    std::vector<unsigned char> w(bytes * L);
    for (size_t b = 0; b < w.size(); b += 36) {
        const float s = 0.002f;
        memcpy(&w[b], &s, 4);
        for (int i = 4; i < 36; i++) w[b + i] = (unsigned char)(int)(100 * uni());
    }
    std::vector<float> x0(NB * D), ln(L * D), kv0((size_t)NB * L * 2 * MS * KV);
    for (float& v : x0) v = uni();
    for (float& v : ln) v = 1 + 0.1f * uni();
    for (float& v : kv0) v = uni();
    a.w = w.data();
    a.ln1 = a.ln2 = ln.data();
    for (int i = 0; i < 32; i++) a.inv_freq[i] = powf(10000.f, -(float)i / 32);
    a.scale = 0.125f;
    a.eps = 1e-5f;
    a.D = D, a.H = H, a.NH = NH, a.NKV = NKV, a.HD = 64, a.KV = KV, a.QD = QD, a.MS = MS, a.L = L;
    a.NB = NB, a.G = 1, a.nch = dec_persist_nch(NKV, NB);
    a.fault_wg = -1;
    a.ex_stride = DEC_PERSIST_EX_WORDS_NB(D, H, QD, KV, NH, 64, NB, a.nch);
    std::vector<float> x, kv, xr, kvr;
    int runs = 0, differ = 0;
    for (int late = -1; late < DEC_PERSIST_WGS * emu::NWAVE; late = late < 0 ? first : late + step) { /* -1: none */
        x = x0;
        kv = kv0;
        std::vector<unsigned long long> ex(a.ex_stride, 0);
        ex[0] = 1;
        DecState st;
        memset(&st, 0, sizeof st);
        st.pos = pos;
        a.x = x.data();
        a.kvc = kv.data();
        a.ex = ex.data();
        a.st = &st;
        emu::late_group = late < 0 ? -1 : late / emu::NWAVE;
        emu::late_wave = late % emu::NWAVE;
        if (dec_launch_persist(&a, nullptr) || emu::stuck || st.sync_error) {
            printf("stuck: wave %d of workgroup %d held back\n", emu::late_wave, emu::late_group);
            return 2;
        }
        if (late < 0) {
            xr = x;
            kvr = kv;
            for (float v : x)
                if (!(fabsf(v) < 1e3f) || x == x0) return 2;
            continue;
        }
        runs++;
        if (memcmp(x.data(), xr.data(), 4 * x.size()) || memcmp(kv.data(), kvr.data(), 4 * kv.size())) {
            differ++;
            printf("differs: wave %d of workgroup %d held back\n", emu::late_wave, emu::late_group);
        }
    }
    printf("runs %d differ %d\n", runs, differ);
    return differ != 0;
}
