// Cooperative row-block solve of long contiguous systems: up to 64 * NW blocks per
// system, the block interfaces solved by merges across lanes.
//
// The schedule and the publication protocol are coop_kernel's (tri_coop.hpp): K
// workgroups hold the K row blocks of one system on chip, each publishes its block's
// outer form and takes the others', so HBM sees 5 words per unknown instead of the
// chunked solve's 9.  With hundreds of blocks a serial chain over them would take tens
// of microseconds; here
//   - the wave-blocks of a block are merged by log2(NW) Wang-Mou rounds across lanes,
//     which gives the block's form and, kept in LDS, each wave-block's ends in terms of
//     the block's neighbours;
//   - lane t of a workgroup polls block t's flag (each wave its own 64 blocks), loads
//     that block's form into registers, and 6 rounds across the wave's lanes plus
//     log2(NW) rounds over the waves' merged forms give x at every block boundary.
//
// Waits are bounded here too: with hundreds of blocks per system a workgroup whose partners
// do not publish waits a bounded number of polls, then leaves its block unsolved (x is not
// written, d is intact) and goes on: every block's form is published in the end, no
// wait depends on a workgroup that cannot run, and coop_mend_kernel, launched after it,
// solves the blocks that were left.  It reads one word per block when there are none.
#pragma once
#include "tri_coop.hpp"

namespace tri {

// Contiguous blocks: whole 16-byte chunks of the wave's 64*M rows, issued
// unconditionally (the buffer ends at the system's last row, so chunks past it
// read as zero).
template <typename T, int M, bool NT>
__device__ __forceinline__ void contig_block_issue(const __amdgpu_buffer_rsrc_t (&rr)[4], int64_t wrow,
                                                   int lane, u32x4 (&g)[4][M * (int)sizeof(T) / 16]) {
    constexpr int NQ = M * (int)sizeof(T) / 16;
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k)
            g[k][q] = load16<NT>(rr[k], (int)(wrow * (int64_t)sizeof(T)) + lane * 16 + q * 1024);
}

template <typename T, int M>
__device__ __forceinline__ void contig_block_transpose(const u32x4 (&g)[4][M * (int)sizeof(T) / 16],
                                                       int lane, u32x4 *xb, T (&rows)[4][M]) {
    constexpr int VV = 16 / (int)sizeof(T);
    constexpr int NQ = M / VV;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (k > 0) wave_lds_sync();
#pragma unroll
        for (int q = 0; q < NQ; ++q) xb[q * 64 + lane] = g[k][q];
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const u32x4 t = xb[lane * NQ + i];
#pragma unroll
            for (int v = 0; v < VV; ++v) rows[k][i * VV + v] = reinterpret_cast<const T *>(&t)[v];
        }
    }
}

// Stores x of the wave's 64*M rows the same way (the buffer drops rows past the system).
template <typename T, int M, bool NT>
__device__ __forceinline__ void contig_block_store(__amdgpu_buffer_rsrc_t rd, int64_t wrow,
                                                   int lane, u32x4 *xb, const T (&xs)[M]) {
    constexpr int VV = 16 / (int)sizeof(T);
    constexpr int NQ = M / VV;
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        u32x4 t;
#pragma unroll
        for (int v = 0; v < VV; ++v) reinterpret_cast<T *>(&t)[v] = xs[i * VV + v];
        xb[lane * NQ + i] = t;
    }
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        store16<NT>(xb[q * 64 + lane], rd, (int)(wrow * (int64_t)sizeof(T)) + lane * 16 + q * 1024);
}

template <typename T, int M, int NW> struct CoopTreeLds {
    u32x4 x[NW][64 * M * (int)sizeof(T) / 16];
    T wave[NW][6];      // wave-blocks' outer forms: first row r, p, q, last row r, p, q
    T merged[NW][6];    // the same relative to the block's neighbours
    T group[NW][6];     // forms of 64 blocks merged by one wave
    T ends[2];          // x of the rows before and after the block
    int ok[NW];
};

template <typename T>
__device__ __forceinline__ void put_form(T *f, const Outer<T> &F, const Outer<T> &E) {
    f[0] = F.r; f[1] = F.p; f[2] = F.q; f[3] = E.r; f[4] = E.p; f[5] = E.q;
}

// Block `task`: loads, reduces and (MEND = false) publishes it, takes the other blocks'
// forms and stores x.  Returns whether x was stored (uniform over the workgroup).
template <typename T, int M, int NW, bool MEND>
__device__ __forceinline__ bool coop_tree_block(const CoopParams<T> &p, int task,
                                                CoopTreeLds<T, M, NW> &lds) {
    using Sh = TileShape<T, M, NW, 1, false, true, false, false, true, true, true>;
    constexpr int R = 64 * NW * M;
    constexpr int NQ = M * (int)sizeof(T) / 16;
    // an opaque copy: lane-dependent addresses and masks stay inside the task loop
    // instead of occupying registers across it
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, ws = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = p.K;
    const int gi = task / K, j = task - gi * K;
    const int64_t brow = (int64_t)j * R, wrow = (int64_t)ws * 64 * M;
    // buffers from the block's first row to the system's last row
    const int64_t base = (int64_t)gi * p.sstride + brow;
    const int32_t bytes = (int32_t)((p.n - brow) * (int64_t)sizeof(T));
    const __amdgpu_buffer_rsrc_t rr[4] = {make_rsrc(p.a + base, bytes), make_rsrc(p.b + base, bytes),
                                          make_rsrc(p.c + base, bytes), make_rsrc(p.d + base, bytes)};
    T rows[4][M];
    {
        u32x4 g[4][NQ];
        contig_block_issue<T, M, true>(rr, wrow, lane, g);
        contig_block_transpose<T, M>(g, lane, lds.x[ws], rows);
    }
#pragma unroll
    for (int q = 0; q < M; ++q)
        if (brow + wrow + lane * M + q >= p.n) {   // identity rows past the system
            rows[0][q] = 0; rows[1][q] = 1; rows[2][q] = 0; rows[3][q] = 0;
        }
    // al is only read back in the substitution: it waits in the wave's transposition
    // block ([row][lane]), which is free until the stores
    T *al = reinterpret_cast<T *>(lds.x[ws]) + lane;
    wave_lds_sync();
    SweepOut<T, Sh::NI> o;
    RegLoader<T, Sh::CH, M> ld{rows};
    lane_sweep<T, Sh>(o, ld, brow + wrow + (int64_t)lane * M, p.n, [&](int q, T x) { al[64 * q] = x; });
    Outer<T> oL, oR;
    {
        const T DLr = o.bL - o.cL * o.SA, ELr = o.cL * o.PI, FLr = o.dL - o.cL * o.SD;
        const T ARr = -(o.aR * o.alp), DRr = o.bR - o.aR * o.g, FRr = o.dR - o.aR * o.del;
        segment_outer(o.aL, DLr, ELr, FLr, ARr, DRr, o.cR, FRr, oL, oR);
    }
    wm_wave_merges<T, 64, 1>(oL, oR, lane, 0, lane, 64, false, nullptr);
    if (lane == 0) { lds.wave[ws][0] = oL.r; lds.wave[ws][1] = oL.p; lds.wave[ws][2] = oL.q; }
    if (lane == 63) { lds.wave[ws][3] = oR.r; lds.wave[ws][4] = oR.p; lds.wave[ws][5] = oR.q; }
    __syncthreads();
    // one array per value of the forms, so that 64 lanes read 64 blocks' as whole lines
    T *fg = p.forms + (int64_t)gi * K * 6;
    uint64_t *flags = p.flags + (int64_t)gi * K;
    if (tid < NW) {
        const T *f = lds.wave[tid];
        Outer<T> F{f[0], f[1], f[2]}, E{f[3], f[4], f[5]};
        wm_wave_merges<T, NW, 1>(F, E, tid, 0, tid, NW, false, nullptr);
        put_form(lds.merged[tid], F, E);
        if constexpr (!MEND) {
            T *out = fg + (int64_t)(tid == 0 ? 0 : 3) * K + j;
            const T v[3] = {tid == 0 ? F.r : E.r, tid == 0 ? F.p : E.p, tid == 0 ? F.q : E.q};
            if (tid == 0 || tid == NW - 1) {
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    __hip_atomic_store(out + (int64_t)q * K, v[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            // both lanes are of wave 0: the form has reached the agent-coherent level
            // before its flag is written (the fences only hold the compiler)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_s_waitcnt(0);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            if (tid == 0)
                __hip_atomic_store(flags + j, p.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // block tid's form; blocks past the last are zero (they pass nothing on)
    Outer<T> F{0, 0, 0}, E{0, 0, 0};
    bool ok = true;
    if (ws * 64 < K) {
        if constexpr (!MEND) {
            bool seen = tid >= K;
            for (int polls = 0;; ++polls) {
                if (!seen)
                    seen = __hip_atomic_load(flags + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.tag;
                if (__all(seen)) break;
                if (polls >= p.spin_limit) { ok = false; break; }
                __builtin_amdgcn_s_sleep(TRI_COOP_POLL_SLEEP);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (ok && tid < K) {
            T f[6];
#pragma unroll
            for (int q = 0; q < 6; ++q)
                f[q] = __hip_atomic_load(fg + (int64_t)q * K + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            F = {f[0], f[1], f[2]};
            E = {f[3], f[4], f[5]};
        }
        wm_wave_merges<T, 64, 1>(F, E, lane, 0, lane, 64, false, nullptr);
    }
    if (lane == 0) {
        lds.group[ws][0] = F.r; lds.group[ws][1] = F.p; lds.group[ws][2] = F.q;
        lds.ok[ws] = ok;
    }
    if (lane == 63) { lds.group[ws][3] = E.r; lds.group[ws][4] = E.p; lds.group[ws][5] = E.q; }
    __syncthreads();
    // x before and after this wave's 64 blocks, from the waves' merged forms
    T u = 0, v = 0;
    {
        const T *f = lds.group[lane < NW ? lane : 0];
        Outer<T> GF{f[0], f[1], f[2]}, GE{f[3], f[4], f[5]};
        wm_wave_merges<T, NW, 1>(GF, GE, lane, 0, lane & (NW - 1), NW, false, nullptr);
        const T ue = lane_read(GE.r, ws > 0 ? ws - 1 : 0), vf = lane_read(GF.r, ws < NW - 1 ? ws + 1 : 0);
        u = ws > 0 ? ue : T(0);
        v = ws < NW - 1 ? vf : T(0);
    }
    if (tid == j - 1) lds.ends[0] = E.r - E.p * u - E.q * v;
    if (tid == j + 1) lds.ends[1] = F.r - F.p * u - F.q * v;
    if (tid == j && j == 0) lds.ends[0] = 0;
    if (tid == j && j == K - 1) lds.ends[1] = 0;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) ok = ok && lds.ok[w] != 0;
    if (!ok) return false;
    const T U = lds.ends[0], V = lds.ends[1];
    u = U;
    v = V;
    if (ws > 0) u = lds.merged[ws - 1][3] - lds.merged[ws - 1][4] * U - lds.merged[ws - 1][5] * V;
    if (ws < NW - 1) v = lds.merged[ws + 1][0] - lds.merged[ws + 1][1] * U - lds.merged[ws + 1][2] * V;
    T xs[M];
    xs[0] = oL.r - oL.p * u - oL.q * v;
    xs[M - 1] = oR.r - oR.p * u - oR.q * v;
    T xn = xs[M - 1];
#pragma unroll
    for (int q = M - 3; q >= 0; --q) {
        xn = (o.de[q] - al[64 * q] * xs[0]) - o.ga[q] * xn;
        xs[q + 1] = xn;
    }
    contig_block_store<T, M, true>(make_rsrc(p.x + base, bytes), wrow, lane, lds.x[ws], xs);
    return true;
}

// p.done[task] takes the solve's tag once x of the block is stored.
template <typename T, int M, int NW, int OCC>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(OCC)))
    coop_tree_kernel(CoopParams<T> p) {
    __shared__ CoopTreeLds<T, M, NW> lds;
    const int ntask = p.ngroups * p.K;
    for (int task = (int)blockIdx.x; task < ntask; task += (int)gridDim.x)
        if (coop_tree_block<T, M, NW, false>(p, task, lds) && threadIdx.x == 0)
            p.done[task] = p.tag;
}

// Solves the blocks whose wait gave up; every block's form is published by now.
template <typename T, int M, int NW, int OCC>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(OCC)))
    coop_mend_kernel(CoopParams<T> p) {
    __shared__ CoopTreeLds<T, M, NW> lds;
    const int ntask = p.ngroups * p.K, P = (int)gridDim.x;
    // one load per lane looks at every block of this workgroup first
    bool left = false;
    for (int64_t t = blockIdx.x + (int64_t)P * threadIdx.x; t < ntask; t += (int64_t)P * 64 * NW)
        left = left || p.done[t] != p.tag;
    if (!__syncthreads_or(left)) return;
    for (int task = (int)blockIdx.x; task < ntask; task += P)
        if (p.done[task] != p.tag) coop_tree_block<T, M, NW, true>(p, task, lds);
}

}  // namespace tri
