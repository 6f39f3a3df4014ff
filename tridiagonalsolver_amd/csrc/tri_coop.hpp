// Cooperative row-block solve: a group of systems whose rows are too many for
// one workgroup is cut into K row blocks, and K workgroups solve the group
// together, each keeping its own block on chip from load to store (5 words of
// HBM traffic per unknown).
//
// This file: interleaved systems, and what both layouts share.  Contiguous systems:
// tri_coop_tree.hpp.
//
//   task (g, j) = rows [j*R, (j+1)*R) of the S systems of group g
//     1. the block's rows (whole row pieces of S*sizeof(T) bytes) go to the lanes
//        through LDS; lane sweeps and Wang-Mou merges inside each wave and across the
//        waves give the block's first row F and last row E in outer form relative to
//        U = x of the row before the block and V = x of the row after it, and the same
//        for every wave-block's ends
//     2. those 6 values per system are published, and the workgroup waits until the
//        other K-1 blocks of the group have published theirs
//     3. partial elimination over the block forms on either side of the block gives U
//        and V, with them the wave-blocks' ends, and the lanes back-substitute from
//        registers and store x
//
// Schedule: the grid is P workgroups, all resident at once (P is at most what the
// device holds, and a multiple of K), and workgroup w takes tasks w, w + P,
// w + 2P, ...  The K tasks of a slot are consecutive, so they fall in the same
// round and every member publishes before it waits: with all P workgroups
// resident, every wait ends.  The slots of a round take groups spread over the whole
// batch (coop_group), so that a round reads whole interleaved rows rather than a strip.
//
// Nothing rests on that.  Other kernels (a large solve on a second stream), or a stream
// that may use only some of the CUs, can keep workgroups of this grid out, and with eight
// XCDs that fill each at its own pace those that run need not hold one whole group.  So
// every wait is bounded (spin_limit polls): a workgroup whose wait gives up publishes its
// remaining tasks without waiting and then finishes them alone (coop_alone): it reduces the
// blocks of a group that are not published and publishes them in their owners' place.  x of
// a block is only ever written by its owner, so every solve ends with every row solved,
// whichever workgroups can run.
//
// Publication without L2 writeback or invalidate: the block forms are written
// with agent-scope atomic stores (which write through to the level where all
// XCDs meet), the writing lanes wait until those stores have completed
// (s_waitcnt) before the workgroup barrier, and one lane then stores the solve's
// tag into the block's flag word with an agent-scope atomic store.  The waiting
// side polls the group's flag words with agent-scope atomic loads and reads the
// forms with agent-scope atomic loads too, so no stale copy in an L1 or L2 can
// serve them.  Tagged flags instead of an arrival counter: nothing has to be
// cleared before a solve (a counter needed a reset kernel per solve, 2-6 us).  An
// acquire/release pair at agent scope would also order them, but it compiles to
// an L2 writeback (release) and invalidate (acquire) per workgroup and task,
// which the XCDs' L2s serve one at a time: measured on MI355X, FP32 interleaved
// 4096 x 4096 took 242 us with them and 175 us without (both before the polls
// were spread over separate lines and the schedule was made static).
//
// The reference has no counterpart: its solvers stream one system through one
// warp (Tridiagonal_CUDA/tridiagonal_wm_pcr.cu:17-205) or reduce in global
// memory level by level (tridiagonal_basic.cu:32-164).
#pragma once
#include "tri_coop_sched.hpp"
#include "tri_tile.hpp"

namespace tri {

template <typename T> struct CoopParams {
    const T *a, *b, *c, *d;
    T *x;                // the solution; d itself, or an array apart from all inputs
    int64_t n, batch;
    int64_t sstride;     // elements between consecutive systems (interleaved: 1)
    int64_t rstride;     // elements between consecutive rows (contiguous: 1)
    int32_t buf_bytes;   // byte extent of each array (below 2 GiB)
    int32_t K;           // row blocks per system
    int32_t ngroups;     // groups of S systems
    int32_t spin_limit;  // polls of a wait before it gives up
    int32_t pipelined;   // 1: coop_pipe_kernel (wait one task later), 0: coop_kernel
    int32_t spread;      // groups per round whose slots are spread over the batch (<= 1: none)
    int32_t shared_lines;  // interleaved rows start off 128-byte lines (coop_task_shared)
    T *forms;            // [ngroups][K][6][S] block outer forms
    uint64_t *flags;     // [kCoopFlagStride * g + j]: the tag once block j of group g is published
    uint64_t tag;        // this solve's tag: different from every earlier solve's
    uint64_t *done;      // coop_tree_kernel: the tag once block t of the grid is solved
};

// Publication flags: one 8-byte word per block of a group (up to 64 blocks), the
// group's words in 512 bytes of their own (so that the polls of different groups
// go to different memory channels).  A block is published when its word holds the
// solve's tag.  Tags never repeat (a 64-bit sequence from a random start), so
// words left by earlier solves, or never written, do not read as published and
// the flags need no clearing between solves.
constexpr int kCoopFlagStride = 64;
// Polls of one wait before it gives up: about 1 ms, where a wait takes microseconds unless
// workgroups of the grid cannot run.
constexpr int kCoopPolls = 1024;
// s_sleep argument between two polls of a wait (64 clocks per unit).
#ifndef TRI_COOP_POLL_SLEEP
#define TRI_COOP_POLL_SLEEP 8
#endif

// Group and row block of an interleaved task.
template <typename T>
__device__ __forceinline__ void coop_task(const CoopParams<T> &p, int task, int &gi, int &j) {
    if (p.shared_lines) {
        coop_task_shared(task, (int)gridDim.x, p.K, p.ngroups, gi, j);
    } else {
        const int s = task / p.K;
        j = task - s * p.K;
        gi = coop_group(s, p.ngroups, p.spread);
    }
}

template <typename T, int M, int NW, int S> struct CoopShape {
    static constexpr int SW = 64 / S;                // segments of a system per wave
    static constexpr int R = SW * NW * M;            // rows per block
};

// Wave 0 of a workgroup waits until all K blocks of group g carry the solve's tag:
// lane k polls block k's word, and the wave goes on once every lane has seen it
// (one vote per poll; its own block's word among them, so that the workgroup's flag is
// known to be visible before it stores x).  Returns 0 if spin_limit polls pass first.
template <typename T>
__device__ __forceinline__ int coop_wait(const CoopParams<T> &p, int g, int lane) {
    const uint64_t *f = p.flags + kCoopFlagStride * g;
    for (int polls = 0;; ++polls) {
        const bool seen =
            lane >= p.K || __hip_atomic_load(f + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.tag;
        if (__all(seen)) return 1;
        if (polls >= p.spin_limit) return 0;
        __builtin_amdgcn_s_sleep(TRI_COOP_POLL_SLEEP);
    }
}

// Forms are kept value by value, [block][6][S], in global memory and in LDS: the S lanes
// that handle one value of a block are consecutive, so global accesses coalesce and LDS
// accesses hit distinct banks.  ([system][block][6], strides of 6 * KMAX words, put the
// lanes of every access of the chain on one LDS bank.)
//
// Stages the K block forms of a group (K*6*S values at fg) into sh_k with the whole
// workgroup.  Each thread issues several loads before it stores the first: the loads are
// agent-scope (they go past the XCD's L2 to where all XCDs meet), and one after another
// their latencies add up.
template <typename T, int S, int NW>
__device__ __forceinline__ void coop_stage_forms(const T *fg, int K, int tid, T *sh_k) {
    constexpr int NT = 64 * NW, B = sizeof(T) == 4 ? 8 : 4;
    const int ne = K * 6 * S;
    for (int e0 = 0; e0 < ne; e0 += NT * B) {
        T v[B];
#pragma unroll
        for (int i = 0; i < B; ++i) {
            const int e = e0 + i * NT + tid;
            v[i] = e < ne ? __hip_atomic_load(fg + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                          : T(0);
        }
#pragma unroll
        for (int i = 0; i < B; ++i) {
            const int e = e0 + i * NT + tid;
            if (e < ne) sh_k[e] = v[i];
        }
    }
}

// x of the rows before (ends[0][s]) and after (ends[1][s]) block j of every system, from the
// K staged block forms.  Lane s eliminates blocks 0 .. j-1, lane S + s blocks K-1 .. j+1 (the
// same recurrence with first and last rows, p and q exchanged): x at the near end of what
// is eliminated is rho - sig * (x at the facing end of the next block).  Block j's own form
// closes the two relations.
template <typename T, int S>
__device__ __forceinline__ void coop_block_ends(const T *k6, int K, int j, int tid, T (*ends)[S]) {
    static_assert(2 * S <= 64, "both sides of a system in one wave");
    if (tid >= 2 * S) return;
    const int s = tid % S;
    const bool right = tid >= S;
    const int steps = right ? K - 1 - j : j;
    const int far = right ? 3 : 0, near = 3 - far, po = right ? 2 : 1, qo = 3 - po;
    const T *f = k6 + (right ? (K - 1) * 6 * S : 0) + s;
    const int df = right ? -6 * S : 6 * S;
    T rho = 0, sig = 0;
    T a[6], b[6];
    auto load = [&](T (&v)[6], const T *g) {
        v[0] = g[far * S]; v[1] = g[(far + po) * S]; v[2] = g[(far + qo) * S];
        v[3] = g[near * S]; v[4] = g[(near + po) * S]; v[5] = g[(near + qo) * S];
    };
    if (steps > 0) load(a, f);
    for (int t = 0; t < steps; ++t) {
        f += df;
        if (t + 1 < steps) load(b, f);
        const T inv = rcp(T(1) - a[1] * sig);
        const T rhoF = (a[0] - a[1] * rho) * inv, sigF = a[2] * inv;
        rho = a[3] - a[4] * (rho - sig * rhoF);
        sig = a[5] + a[4] * sig * sigF;
#pragma unroll
        for (int q = 0; q < 6; ++q) a[q] = b[q];
    }
    const T rhoR = lane_read(rho, S + s), sigR = lane_read(sig, S + s);
    if (right) return;
    const T *o = k6 + j * 6 * S + s;
    const T pF = o[S], qF = o[2 * S], pE = o[4 * S], qE = o[5 * S];
    const T bF = o[0] - pF * rho - qF * rhoR, bE = o[3 * S] - pE * rho - qE * rhoR;
    const T mFF = T(1) - pF * sig, mFE = qF * sigR, mEF = pE * sig, mEE = T(1) - qE * sigR;
    const T inv = rcp(mFF * mEE - mFE * mEF);
    ends[0][s] = rho - sig * ((mEE * bF + mFE * bE) * inv);
    ends[1][s] = rhoR - sigR * ((mEF * bF + mFF * bE) * inv);
}

// Wave-blocks' forms of a task in LDS, [wave][6][S] with the waves SG apart in the banks.
template <typename T, int NW, int S> struct CoopWaveForms {
    static constexpr int SG = 64 / NW;             // systems whose waves one wave merges
    static_assert(NW * SG == 64 && S % SG == 0, "a wave merges whole systems");
    T v[NW][6 * S + SG];
};

template <typename T>
__device__ __forceinline__ void coop_rsrc(const CoopParams<T> &p, __amdgpu_buffer_rsrc_t (&rr)[4]) {
    rr[0] = make_rsrc(p.a, p.buf_bytes); rr[1] = make_rsrc(p.b, p.buf_bytes);
    rr[2] = make_rsrc(p.c, p.buf_bytes); rr[3] = make_rsrc(p.d, p.buf_bytes);
}

// Publishes a task's block form.  The waves' forms (oL, oR after the merges inside each
// wave) meet in LDS and log2(NW) merges across lanes give each wave-block's ends in terms
// of the block's neighbours, which stay in wf for coop_finish; the first and last of them
// are the block's form.  ALONE: without publishing.
template <typename T, int NW, int S, bool ALONE = false>
__device__ __forceinline__ void coop_publish(const CoopParams<T> &p, int gi, int j,
                                             const Outer<T> &oL, const Outer<T> &oR, int tid,
                                             CoopWaveForms<T, NW, S> &wf) {
    constexpr int SW = 64 / S, SG = CoopWaveForms<T, NW, S>::SG;
    const int lane = tid & 63, wave = tid >> 6, sl = lane % S, kw = lane / S;
    T *f = wf.v[wave] + sl;
    if (kw == 0) { f[0] = oL.r; f[S] = oL.p; f[2 * S] = oL.q; }
    if (kw == SW - 1) { f[3 * S] = oR.r; f[4 * S] = oR.p; f[5 * S] = oR.q; }
    __syncthreads();
    if (tid < S * NW) {
        const int s = wave * SG + lane % SG, w = lane / SG;
        T *m = wf.v[w] + s;
        Outer<T> F{m[0], m[S], m[2 * S]}, E{m[3 * S], m[4 * S], m[5 * S]};
        wm_wave_merges<T, NW, SG>(F, E, lane, lane % SG, w, NW, false, nullptr);
        m[0] = F.r; m[S] = F.p; m[2 * S] = F.q;
        m[3 * S] = E.r; m[4 * S] = E.p; m[5 * S] = E.q;
        if (!ALONE && (w == 0 || w == NW - 1)) {
            T *out = p.forms + (((int64_t)gi * p.K + j) * 6 + (w == 0 ? 0 : 3)) * S + s;
            const T v[3] = {w == 0 ? F.r : E.r, w == 0 ? F.p : E.p, w == 0 ? F.q : E.q};
#pragma unroll
            for (int q = 0; q < 3; ++q)
                __hip_atomic_store(out + q * S, v[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // the forms are at the agent-coherent level before the barrier
        if (!ALONE) __builtin_amdgcn_s_waitcnt(0);
    }
    __syncthreads();
    if (!ALONE && tid == 0)
        __hip_atomic_store(p.flags + kCoopFlagStride * gi + j, p.tag, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}

// Large LDS buffer of a task: the waves' transposition blocks while rows and x move, the
// group's block forms in between (64 blocks' forms still leave two workgroups per CU).
template <typename T, int M, int NW, int S, int KMAX> struct CoopBuf {
    static constexpr int kRows = NW * 64 * M * (int)sizeof(T) / 16;
    static constexpr int kForms = KMAX * 6 * S * (int)sizeof(T) / 16;
    u32x4 v[kRows > kForms ? kRows : kForms];
    __device__ __forceinline__ u32x4 *wave(int w) { return v + w * (64 * M * (int)sizeof(T) / 16); }
    __device__ __forceinline__ T *forms() { return reinterpret_cast<T *>(v); }
};
template <typename T, int S> struct CoopEnds {
    T x[2][S];      // x before and after the block
    int ok;
};

// Back-substitution of one task once its group has published: waits for the K block forms
// of group gi, takes x around block j from them, x around every wave-block from wf, and
// stores x of the block.  Returns false, with nothing stored, where the wait gave up (the same
// for the whole workgroup).  ALONE: all forms are published, no wait.
template <typename T, int M, int NW, int S, int KMAX, int NI, bool ALONE = false>
__device__ __forceinline__ bool coop_finish(const CoopParams<T> &p, int gi, int j,
                                            const CoopWaveForms<T, NW, S> &wf,
                                            CoopBuf<T, M, NW, S, KMAX> &buf, CoopEnds<T, S> &ends, int tid,
                                            const Outer<T> &oL, const Outer<T> &oR,
                                            const T (&de)[NI], const T (&ga)[NI],
                                            const T (&al)[NI]) {
    constexpr int SW = 64 / S;
    constexpr int R = SW * NW * M;
    const int lane = tid & 63, ws = tid >> 6, sl = lane % S, kw = lane / S;
    if constexpr (!ALONE) {
        if (tid < 64) {
            const int ok = coop_wait(p, gi, tid);
            if (tid == 0) ends.ok = ok;
        }
        __syncthreads();
        if (!ends.ok) return false;
    }
    coop_stage_forms<T, S, NW>(p.forms + (int64_t)gi * p.K * 6 * S, p.K, tid, buf.forms());
    __syncthreads();
    coop_block_ends<T, S>(buf.forms(), p.K, j, tid, ends.x);
    __syncthreads();
    const T U = ends.x[0][sl], V = ends.x[1][sl];
    T u = U, v = V;
    if (ws > 0) {
        const T *f = wf.v[ws - 1] + 3 * S + sl;
        u = f[0] - f[S] * U - f[2 * S] * V;
    }
    if (ws < NW - 1) {
        const T *f = wf.v[ws + 1] + sl;
        v = f[0] - f[S] * U - f[2 * S] * V;
    }
    const T xL = oL.r - oL.p * u - oL.q * v;
    const T xR = oR.r - oR.p * u - oR.q * v;
    T xs[M];
    xs[0] = xL;
    xs[M - 1] = xR;
    T xn = xR;
#pragma unroll
    for (int q = M - 3; q >= 0; --q) {
        xn = (de[q] - al[q] * xL) - ga[q] * xn;
        xs[q + 1] = xn;
    }
    il_block_store<T, M, SW, S, true, true>(make_rsrc(p.x, p.buf_bytes),
                                            (int64_t)j * R + (int64_t)ws * SW * M, p.rstride,
                                            (int64_t)gi * S, p.n, p.batch, lane, sl, kw, buf.wave(ws), xs);
    __syncthreads();                           // LDS of this task free
    return true;
}

// Sweep of the lane's M rows (row0 = its first) and the merges inside the wave: the lane's
// ends in outer form relative to the wave-block's neighbours.
template <typename T, class Sh, int M, int S>
__device__ __forceinline__ void coop_reduce(const T (&rows)[4][M], int64_t row0, int64_t n, int lane,
                                            SweepOut<T, Sh::NI> &o, T (&al)[Sh::NI], Outer<T> &oL,
                                            Outer<T> &oR) {
    RegLoader<T, Sh::CH, M> ld{rows};
    lane_sweep<T, Sh>(o, ld, row0, n, [&](int q, T x) { al[q] = x; });   // drops a_0 and c_{n-1}
    const T DLr = o.bL - o.cL * o.SA, ELr = o.cL * o.PI, FLr = o.dL - o.cL * o.SD;
    const T ARr = -(o.aR * o.alp), DRr = o.bR - o.aR * o.g, FRr = o.dR - o.aR * o.del;
    segment_outer(o.aL, DLr, ELr, FLr, ARr, DRr, o.cR, FRr, oL, oR);
    wm_wave_merges<T, 64 / S, S>(oL, oR, lane, lane % S, lane / S, 64 / S, false, nullptr);
}

// A task after a wait gave up: the unpublished blocks of its group are reduced and
// published here, then its own block is reduced again and finished without a wait.  In place, the
// owner of a block stores x over the d that is read here, but only after its flag is visible:
// the flag is looked at once the block has been read, and where it is set the owner's form
// stands and this one is dropped.  Otherwise both write the same values.  Runs after the
// task loop, for the task whose wait gave up and those after it, which only published: inside
// the loop it cost registers (FP64 3001 x 1001 33.5 / 34.1 us).
template <typename T, int M, int NW, int S, int KMAX>
__device__ __forceinline__ void coop_alone(const CoopParams<T> &p, int task,
                                           CoopWaveForms<T, NW, S> &wf,
                                           CoopBuf<T, M, NW, S, KMAX> &buf, CoopEnds<T, S> &ends) {
    using Sh = TileShape<T, M, NW, S, true, false, false, false, false, true, true>;
    constexpr int SW = 64 / S, R = SW * NW * M;
    int gi, j;
    coop_task(p, task, gi, j);
    uint64_t *flags = p.flags + kCoopFlagStride * gi;
    auto published = [&](int k) {              // the same answer for the whole workgroup
        __syncthreads();
        if (threadIdx.x == 0)
            ends.ok = __hip_atomic_load(flags + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.tag;
        __syncthreads();
        return ends.ok != 0;
    };
    for (int k = 0; k <= p.K; ++k) {           // block j itself is published; it comes last
        const bool own = k == p.K;
        if (!own && published(k)) continue;
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, wave = tid >> 6, sl = lane % S, kw = lane / S;
        const int64_t wrow = (int64_t)(own ? j : k) * R + (int64_t)wave * SW * M;
        __amdgpu_buffer_rsrc_t rr[4];
        coop_rsrc(p, rr);
        T rows[4][M], al[Sh::NI];
        il_block_load<T, M, SW, S, false, true>(rr, wrow, p.rstride, (int64_t)gi * S, p.n, lane, sl, kw,
                                                buf.wave(wave), rows);
        SweepOut<T, Sh::NI> o;
        Outer<T> oL, oR;
        coop_reduce<T, Sh, M, S>(rows, wrow + (int64_t)kw * M, p.n, lane, o, al, oL, oR);
        coop_publish<T, NW, S, true>(p, gi, j, oL, oR, tid, wf);
        if (own) {
            coop_finish<T, M, NW, S, KMAX, Sh::NI, true>(p, gi, j, wf, buf, ends, tid, oL, oR, o.de,
                                                         o.ga, al);
        } else if (!published(k)) {
            if (tid < S) {
                T *out = p.forms + ((int64_t)gi * p.K + k) * 6 * S + tid;
#pragma unroll
                for (int q = 0; q < 6; ++q)
                    __hip_atomic_store(out + q * S, wf.v[q < 3 ? 0 : NW - 1][q * S + tid], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                __builtin_amdgcn_s_waitcnt(0);
            }
            __syncthreads();
            if (tid == 0)
                __hip_atomic_store(flags + k, p.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// OCC: waves per SIMD the kernel is built for (its register budget).  LINES: rows start on
// 128-byte lines, which are read once and streamed; otherwise neighbouring groups share
// lines and the loads stay cached.
template <typename T, int M, int NW, int S, int KMAX, int OCC, bool LINES>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(OCC)))
    coop_kernel(CoopParams<T> p) {
    using Sh = TileShape<T, M, NW, S, true, false, false, false, false, true, true>;
    constexpr int SW = 64 / S;               // segments of a system per wave
    constexpr int R = SW * NW * M;           // rows per block
    static_assert((S * (int)sizeof(T)) % 16 == 0, "blocks move whole 16-byte chunks");
    static_assert(KMAX <= kCoopFlagStride, "a group's flags fit its flag words");
    __shared__ CoopBuf<T, M, NW, S, KMAX> buf;
    __shared__ CoopWaveForms<T, NW, S> wf;
    __shared__ CoopEnds<T, S> ends;

    const int P = (int)gridDim.x;
    const int ntask = p.ngroups * p.K;
    int left = ntask;                        // first task whose wait gave up
    for (int task = (int)blockIdx.x; task < ntask; task += P) {
        // an opaque copy: lane-dependent addresses and masks stay inside the task loop
        // instead of occupying registers across it
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, wave = tid >> 6;
        const int sl = lane % S;             // system of the lane inside the group
        const int kw = lane / S;             // segment inside the wave-block
        int gi, j;
        coop_task(p, task, gi, j);
        const int64_t wrow = (int64_t)j * R + (int64_t)wave * SW * M;   // first row of the wave
        __amdgpu_buffer_rsrc_t rr[4];
        coop_rsrc(p, rr);
        T rows[4][M], al[Sh::NI];
        il_block_load<T, M, SW, S, LINES, true>(rr, wrow, p.rstride, (int64_t)gi * S, p.n, lane, sl, kw,
                                                buf.wave(wave), rows);
        SweepOut<T, Sh::NI> o;
        Outer<T> oL, oR;
        coop_reduce<T, Sh, M, S>(rows, wrow + (int64_t)kw * M, p.n, lane, o, al, oL, oR);
        coop_publish<T, NW, S>(p, gi, j, oL, oR, tid, wf);
        if (left == ntask && !coop_finish<T, M, NW, S, KMAX, Sh::NI>(p, gi, j, wf, buf, ends, tid, oL,
                                                                     oR, o.de, o.ga, al))
            left = task;
    }
    for (; left < ntask; left += P) coop_alone<T, M, NW, S, KMAX>(p, left, wf, buf, ends);
}

// The same solve with the wait taken one task later: a workgroup reduces and
// publishes task t + P before it waits for the group of task t, so the time the
// group's slowest member needs is covered by a whole task's loads and arithmetic
// instead of idling.  The lane state of the pending task (its outer forms and the
// sweep coefficients of its rows, 3(M-2) + 6 values per lane) stays in registers.
// Every wait for task t still comes after the workgroup has published task t + P,
// and every member of a group publishes it before waiting on anything later, so
// with all P workgroups resident every wait ends.
template <typename T, int M, int NW, int S, int KMAX>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
    coop_pipe_kernel(CoopParams<T> p) {
    using Sh = TileShape<T, M, NW, S, true, false, false, false, false, true, true>;
    constexpr int SW = 64 / S;
    constexpr int R = SW * NW * M;
    constexpr int NQ = M * (int)sizeof(T) / 16;
    constexpr int NI = Sh::NI;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sl = lane % S;
    const int kw = lane / S;
    const int64_t wrow = (int64_t)wave * SW * M;
    __shared__ CoopBuf<T, M, NW, S, KMAX> buf;
    __shared__ CoopWaveForms<T, NW, S> wf[2];
    __shared__ CoopEnds<T, S> ends;

    const int P = (int)gridDim.x;
    const int ntask = p.ngroups * p.K;
    const int64_t n = p.n;
    int task = (int)blockIdx.x;
    u32x4 g[4][NQ];
    auto issue = [&](int t) {
        int gi, j;
        coop_task(p, t, gi, j);
        __amdgpu_buffer_rsrc_t rr[4];
        coop_rsrc(p, rr);
        il_block_issue<T, M, SW, S, true, true>(rr, (int64_t)j * R + wrow, p.rstride, (int64_t)gi * S,
                                                n, lane, g);
    };
    if (task < ntask) issue(task);
    // the pending task: published, not yet finished
    int pend = -1, par = 0;
    Outer<T> poL{}, poR{};
    T pde[NI], pga[NI], pal[NI];
    int left = ntask;
    auto finish = [&]() {
        int gi, j;
        coop_task(p, pend, gi, j);
        if (left == ntask && !coop_finish<T, M, NW, S, KMAX, NI>(p, gi, j, wf[par ^ 1], buf, ends, tid,
                                                                 poL, poR, pde, pga, pal))
            left = pend;
    };
    for (; task < ntask; task += P) {
        int gi, j;
        coop_task(p, task, gi, j);
        const int64_t row0 = (int64_t)j * R + wrow + (int64_t)kw * M;
        T rows[4][M], al[NI];
        il_block_transpose<T, M, S>(g, lane, sl, kw, buf.wave(wave), rows);
        identity_rows<T, M>(row0, n, rows);
        SweepOut<T, NI> o;
        Outer<T> oL, oR;
        coop_reduce<T, Sh, M, S>(rows, row0, n, lane, o, al, oL, oR);
        coop_publish<T, NW, S>(p, gi, j, oL, oR, tid, wf[par]);
        if (task + P < ntask) issue(task + P);
        if (pend >= 0) finish();
        pend = task;
        par ^= 1;
        poL = oL;
        poR = oR;
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            pde[q] = o.de[q];
            pga[q] = o.ga[q];
            pal[q] = al[q];
        }
    }
    if (pend >= 0) finish();
    for (; left < ntask; left += P) coop_alone<T, M, NW, S, KMAX>(p, left, wf[0], buf, ends);
}

template <typename T> struct CoopEntry {
    int M, NW, S;
    bool IL;     // interleaved: coop_kernel; contiguous: coop_tree_kernel
    int R;       // rows per block
    int kmax;    // most blocks per system (LDS for the block chain)
    bool pipe;   // coop_pipe_kernel by default
    hipError_t (*launch)(const CoopParams<T> &, int grid, hipStream_t);
    int (*max_grid)(bool pipelined);   // co-resident workgroups of the kernel (0: unknown)
};
template <typename T> struct CoopTable {
    const CoopEntry<T> *entries;
    int count;
};
CoopTable<float> coop_table_f32();
CoopTable<double> coop_table_f64();
// Sets `count` words to zero (flags of a solve recorded into a graph).
hipError_t launch_coop_clear(uint64_t *words, int64_t count, hipStream_t st);

}  // namespace tri
