// Adjoint (backward) of the batched solve, and the fused forward + adjoint.
//
// For x = A^{-1} d and an upstream gradient g = dL/dx:
//   lambda = A^{-T} g,  dL/da_i = -lambda_i x_{i-1},  dL/db_i = -lambda_i x_i,
//   dL/dc_i = -lambda_i x_{i+1},  dL/dd_i = lambda_i   (a_0, c_{n-1} are not in A).
// A^T is tridiagonal with sub-diagonal c_{i-1}, diagonal b_i, super-diagonal
// a_{i+1}; it is solved with the same on-chip partition solver as the forward
// problem (lane sweep, interface solve, substitution), fed with the shifted
// coefficients.
//   MODE kAdjoint : reads a, b, c, x, g; writes the four gradients (9 words/row).
//   MODE kFused   : reads a, b, c, d, g; solves A x = d, keeps a, b, c in VGPRs,
//                   solves A^T lambda = g and writes x and the gradients
//                   (10 words/row instead of 14 for a forward and a backward pass).
#pragma once
#include "tri_host.hpp"

namespace tri {

enum AdjMode : int { kAdjoint = 0, kFused = 1 };

template <typename T> struct AdjParams {
    const T *a, *b, *c;
    const T *d;   // kFused: right-hand side; kAdjoint: unused
    const T *x;   // kAdjoint: forward solution; kFused: unused
    const T *g;   // upstream gradient dL/dx
    T *xo;        // kFused: x output
    T *ga, *gb, *gc, *gd;
    int64_t n, batch, sstride, rstride;
    int32_t buf_bytes;
    int32_t iface, xchg_lds;
    int32_t line_tiles = 1;   // interleaved: neighbouring tiles that share lines (launch_adj)
};

// Contiguous layout: a wave's rows [wrow, wrow + 64*M) of one system are read as whole
// 16-byte chunks (consecutive lanes, consecutive chunks; nontemporal).  The descriptor
// spans the system's own rows, so chunks that straddle or pass its end need no predicate
// (the buffer checks each dword: loads past it give zero, stores past it are dropped)
// and rows may start at any element.
template <typename T, int M>
__device__ __forceinline__ void adj_issue(__amdgpu_buffer_rsrc_t r, int64_t wrow, int lane,
                                          u32x4 (&g)[M * (int)sizeof(T) / 16]) {
#pragma unroll
    for (int q = 0; q < M * (int)sizeof(T) / 16; ++q)
        g[q] = load16<true>(r, (int)(wrow * (int64_t)sizeof(T)) + lane * 16 + q * 1024);
}

// Hands every lane its M rows of the chunks in g through the wave's LDS block `xb`, with
// the row before (prev) and after (next) its segment: the neighbouring lanes' rows or,
// at the ends of the block, the given values.
template <typename T, int M>
__device__ __forceinline__ void adj_take(const u32x4 (&g)[M * (int)sizeof(T) / 16], int lane,
                                         u32x4 *xb, T (&rows)[M], T &prev, T &next) {
    constexpr int VV = 16 / (int)sizeof(T);
    constexpr int NQ = M / VV;
    wave_lds_sync();                                  // the block is free
#pragma unroll
    for (int q = 0; q < NQ; ++q) xb[q * 64 + lane] = g[q];
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const u32x4 t = xb[lane * NQ + i];
#pragma unroll
        for (int v = 0; v < VV; ++v) rows[i * VV + v] = reinterpret_cast<const T *>(&t)[v];
    }
    const T *tb = reinterpret_cast<const T *>(xb);
    if (lane > 0) prev = tb[lane * M - 1];
    if (lane < 63) next = tb[lane * M + M];
}

// Writes the lane's M values back as whole 16-byte chunks of the wave block.
template <typename T, int M>
__device__ __forceinline__ void adj_wave_store(__amdgpu_buffer_rsrc_t r, int64_t wrow, int lane,
                                               u32x4 *xb, const T (&vals)[M]) {
    constexpr int VV = 16 / (int)sizeof(T);
    constexpr int NQ = M / VV;
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        u32x4 t;
#pragma unroll
        for (int v = 0; v < VV; ++v) reinterpret_cast<T *>(&t)[v] = vals[i * VV + v];
        xb[lane * NQ + i] = t;
    }
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        store16<true>(xb[q * 64 + lane], r,
                      (int)(wrow * (int64_t)sizeof(T)) + lane * 16 + q * 1024);
}

// Interleaved layout: the same for rows [wrow, wrow + SW*M) of S neighbouring systems, as
// whole row pieces of S*sizeof(T) bytes; rows at or past n lie past the buffer.
template <typename T, int M, int S, bool NT>
__device__ __forceinline__ void adj_il_issue(__amdgpu_buffer_rsrc_t r, int64_t wrow, int64_t rs,
                                             int64_t col0, int64_t n, int lane,
                                             u32x4 (&g)[M * (int)sizeof(T) / 16]) {
    constexpr int CPR = S * (int)sizeof(T) / 16;
#pragma unroll
    for (int q = 0; q < M * (int)sizeof(T) / 16; ++q) {
        const int cidx = q * 64 + lane;
        g[q] = __builtin_amdgcn_raw_buffer_load_b128(
            r, il_chunk_offset<T, true>(wrow + cidx / CPR, rs, col0, n, cidx % CPR), 0, cpol<NT>());
    }
}

template <typename T, int M, int S>
__device__ __forceinline__ void adj_il_take(const u32x4 (&g)[M * (int)sizeof(T) / 16], int lane,
                                            u32x4 *xb, T (&rows)[M], T &prev, T &next) {
    const int sl = lane % S, kw = lane / S;
    wave_lds_sync();                                  // the block is free
#pragma unroll
    for (int q = 0; q < M * (int)sizeof(T) / 16; ++q) xb[q * 64 + lane] = g[q];
    wave_lds_sync();
    const T *tb = reinterpret_cast<const T *>(xb);
#pragma unroll
    for (int j = 0; j < M; ++j) rows[j] = tb[(kw * M + j) * S + sl];
    if (kw > 0) prev = tb[(kw * M - 1) * S + sl];
    if (kw < 64 / S - 1) next = tb[(kw * M + M) * S + sl];
}

// NT: the loads stream (interleaved rows on 128-byte lines; contiguous rows always do).
template <typename T, int M, int NW, int S, bool IL, int MODE, bool NT>
__global__ void __launch_bounds__(64 * NW) tile_adj_kernel(AdjParams<T> prm) {
    using Sh = TileShape<T, M, NW, S, IL, false, false, false, true, false, false>;
    constexpr int SW = Sh::SW, NWS = Sh::NWS, LS = Sh::LS, CH = Sh::CH;
    constexpr int LANES = 64 * NW;
    static_assert((IL ? S : M) * (int)sizeof(T) >= 16, "adjoint tiles move 16-byte chunks");
    extern __shared__ __attribute__((aligned(16))) char tri_dyn_lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int sl = IL ? (lane % S) : (wave / NWS);
    const int kw = IL ? (lane / S) : lane;
    const int ws = IL ? wave : (wave % NWS);
    const int64_t n = prm.n;
    int tile = blockIdx.x;
    if (IL) tile = xcd_group(blockIdx.x, gridDim.x, prm.line_tiles);
    const int64_t sys = (int64_t)tile * S + sl;
    const bool valid = sys < prm.batch;
    const int64_t sysc = valid ? sys : prm.batch - 1;
    const int seg = ws * SW + kw;
    const int64_t row0 = (int64_t)seg * M;

    // raw rows j = 0..M-1 plus the neighbours needed by A^T at the segment edges
    T ra[M], rb[M], rc[M], rg[M], rx[M];
    T c_before, a_after, x_before = 0, x_after = 0;
    __shared__ u32x4 xbuf[NW][64 * M * (int)sizeof(T) / 16];
    // contiguous: per-wave descriptors on the system's own rows (none of an idle wave)
    const int64_t sbase = IL ? 0 : wave_uniform(sysc * n);
    const int32_t sbytes = valid ? (int32_t)(n * (int64_t)sizeof(T)) : 0;
    const int64_t wrow = (int64_t)ws * SW * M;
    auto RW = [&](const T *p) { return make_rsrc(p + sbase, sbytes); };
    // The last array, which only the second half of the work reads (fused: g; adjoint: x),
    // stays in flight during the first solve.  MI355X, taken at once / this (us): FP32 fused
    // 600 x 8000 41.0 / 39.6, 2048 x 2000 33.9 / 32.5, FP64 2000 x 1000 37.0 / 35.3; adjoint
    // FP32 512 x 8192 28.3 / 27.0, 100 x 40,000 35.6 / 33.5, FP64 500 x 4000 29.4 / 28.3.  The
    // adjoint of contiguous systems of several waves does not gain (FP32 2047 x 2048 28.2 /
    // 29.3, FP64 777 x 4000 42.8 / 43.2) and takes x at once.
    constexpr bool kLater = MODE == kFused || IL || NWS == 1;
    u32x4 last[M * (int)sizeof(T) / 16];
    if constexpr (IL) {
        // as below, two arrays in flight; the rows just outside the wave's block are read by
        // the lanes at its ends.  Reading 32-byte pieces one element per lane and row took
        // (us, before / now): FP32 fused 60 x 60,000 50.5 / 32.4, 60 x 59,999 78.2 / 35.4, 448 x
        // 8192 67.4 / 45.9; adjoint FP32 170 x 20,000 42.7 / 25.6, FP64 250 x 8000 69.0 / 35.2
        // (4.1 TB/s).  The fused kernels hold five arrays and two solves in registers, which
        // leaves two or three waves per SIMD.
        constexpr int NQ = M * (int)sizeof(T) / 16;
        const int64_t rs = prm.rstride, col0 = (int64_t)tile * S;
        u32x4 g[4][NQ];
        u32x4 *xb = xbuf[wave];
        T unused = 0;
        auto issue = [&](const T *p, u32x4 (&q)[NQ]) {
            adj_il_issue<T, M, S, NT>(make_rsrc(p, prm.buf_bytes), wrow, rs, col0, n, lane, q);
        };
        auto outside = [&](const T *p, int64_t r, bool end) {
            const int vo = (int)((r * rs + sysc) * (int64_t)sizeof(T));
            return bload<T>(make_rsrc(p, prm.buf_bytes), end && r >= 0 && r < n ? vo : 0x7fffff00, 0);
        };
        issue(prm.b, g[0]);
        issue(prm.c, g[1]);
        c_before = outside(prm.c, wrow - 1, kw == 0);
        a_after = outside(prm.a, wrow + SW * M, kw == SW - 1);
        if constexpr (MODE == kAdjoint) {
            x_before = outside(prm.x, wrow - 1, kw == 0);
            x_after = outside(prm.x, wrow + SW * M, kw == SW - 1);
        }
        adj_il_take<T, M, S>(g[0], lane, xb, rb, unused, unused);
        issue(prm.a, g[2]);
        adj_il_take<T, M, S>(g[1], lane, xb, rc, c_before, unused);
        issue(MODE == kFused ? prm.d : prm.g, g[3]);
        adj_il_take<T, M, S>(g[2], lane, xb, ra, unused, a_after);
        issue(MODE == kFused ? prm.g : prm.x, last);
        adj_il_take<T, M, S>(g[3], lane, xb, MODE == kFused ? rx : rg, unused, unused);
    } else {
        // Two arrays in flight: the next one is issued while the first goes through LDS.
        // The kernel streams, so what counts is that loads never drain: one array at a
        // time and all five at once both lose.  Measured on MI355X, one / two / three /
        // all arrays in flight (us): FP32 fused 512 x 8192 31.8 / 31.9 / 34.0 / 33.0,
        // 100 x 40,000 61.7 / 56.5 / 54.8 / 52.4; adjoint 2047 x 2048 29.8 / 28.4 / 29.6
        // / 30.5, 4096 x 1024 28.5 / 29.5 / 29.7 / 30.8; FP64 adjoint 2048 x 1024 26.5 /
        // 24.3 / 25.2 / 25.3 (6.2 TB/s).  With a predicate per chunk instead of the
        // descriptor's bounds (FP64 adjoint 777 x 4000) 62.0, now 43.0; FP32 2047 x 2048
        // 35.2, now 28.4.
        constexpr int NQ = M * (int)sizeof(T) / 16;
        u32x4 g[4][NQ];
        u32x4 *xb = xbuf[wave];
        T unused = 0;
        adj_issue<T, M>(RW(prm.b), wrow, lane, g[0]);
        adj_issue<T, M>(RW(prm.c), wrow, lane, g[1]);
        c_before = 0;
        a_after = 0;
        if constexpr (NWS > 1) {
            // the rows just outside the block (past an end of the system: zero); through
            // LDS and a barrier they were slower (FP64 1024 x 3000 38.2 / 40.5 us)
            const int before = wrow > 0 ? (int)((wrow - 1) * (int64_t)sizeof(T)) : sbytes;
            const int after = (int)((wrow + 64 * M) * (int64_t)sizeof(T));
            c_before = bload<T>(RW(prm.c), before, 0);
            a_after = bload<T>(RW(prm.a), after, 0);
            if constexpr (MODE == kAdjoint) {
                x_before = bload<T>(RW(prm.x), before, 0);
                x_after = bload<T>(RW(prm.x), after, 0);
            }
        }
        adj_take<T, M>(g[0], lane, xb, rb, unused, unused);
        adj_issue<T, M>(RW(prm.a), wrow, lane, g[2]);
        adj_take<T, M>(g[1], lane, xb, rc, c_before, unused);
        adj_issue<T, M>(RW(MODE == kFused ? prm.d : prm.g), wrow, lane, g[3]);
        adj_take<T, M>(g[2], lane, xb, ra, unused, a_after);
        adj_issue<T, M>(RW(MODE == kFused ? prm.g : prm.x), wrow, lane, last);
        adj_take<T, M>(g[3], lane, xb, MODE == kFused ? rx : rg, unused, unused);
    }
    auto take_last = [&](T (&rows)[M], T &prev, T &next) {
        if constexpr (IL) adj_il_take<T, M, S>(last, lane, xbuf[wave], rows, prev, next);
        else adj_take<T, M>(last, lane, xbuf[wave], rows, prev, next);
    };
    if constexpr (!kLater) take_last(rx, x_before, x_after);
#pragma unroll
    for (int j = 0; j < M; ++j)
        if (row0 + j >= n) rb[j] = 1;                    // identity rows past the end

    T al_r[Sh::NI];
    auto al_store = [&](int j, T v) { al_r[j] = v; };

    // ------------------------------------------------------------ forward (fused)
    if constexpr (MODE == kFused) {
        T rows[4][M];
#pragma unroll
        for (int j = 0; j < M; ++j) {
            rows[0][j] = ra[j]; rows[1][j] = rb[j]; rows[2][j] = rc[j]; rows[3][j] = rx[j];
        }
        SweepOut<T, Sh::NI> o;
        RegLoader<T, CH, M> ld{rows};
        lane_sweep<T, Sh>(o, ld, row0, n, al_store);
        const T DLr = o.bL - o.cL * o.SA, ELr = o.cL * o.PI, FLr = o.dL - o.cL * o.SD;
        const T ARr = -(o.aR * o.alp), DRr = o.bR - o.aR * o.g, FRr = o.dR - o.aR * o.del;
        T xL, xR;
        interface_solve<T, S, SW, NWS, LS, Sh::P, LANES>(o.aL, DLr, ELr, FLr, ARr, DRr, o.cR, FRr,
                                                         tid, lane, sl, kw, ws, prm.iface,
                                                         prm.xchg_lds, tri_dyn_lds, xL, xR);
        rx[0] = xL;
        rx[M - 1] = xR;
        T xn = xR;
#pragma unroll
        for (int j = M - 3; j >= 0; --j) {
            xn = (o.de[j] - al_r[j] * xL) - o.ga[j] * xn;
            rx[j + 1] = xn;
        }
        // x at the rows just outside the segment, from the neighbouring segments
        __shared__ T sh_x[S][2 * Sh::P];
        sh_x[sl][2 * seg] = xL;
        sh_x[sl][2 * seg + 1] = xR;
        __syncthreads();
        x_before = (seg > 0) ? sh_x[sl][2 * seg - 1] : T(0);
        x_after = (seg + 1 < Sh::P) ? sh_x[sl][2 * seg + 2] : T(0);
        __syncthreads();   // interface LDS is reused by the adjoint solve
        T unused = 0;
        take_last(rg, unused, unused);
    }

    // ------------------------------------------------------------ adjoint solve
    T lam[M];
    {
        T rows[4][M];
#pragma unroll
        for (int j = 0; j < M; ++j) {
            rows[0][j] = (j == 0) ? c_before : rc[j - 1];      // sub of A^T: c_{i-1}
            rows[1][j] = rb[j];
            rows[2][j] = (j == M - 1) ? a_after : ra[j + 1];   // super of A^T: a_{i+1}
            rows[3][j] = rg[j];
            if (row0 + j >= n) { rows[0][j] = 0; rows[2][j] = 0; rows[3][j] = 0; }
        }
        SweepOut<T, Sh::NI> o;
        RegLoader<T, CH, M> ld{rows};
        lane_sweep<T, Sh>(o, ld, row0, n, al_store);
        const T DLr = o.bL - o.cL * o.SA, ELr = o.cL * o.PI, FLr = o.dL - o.cL * o.SD;
        const T ARr = -(o.aR * o.alp), DRr = o.bR - o.aR * o.g, FRr = o.dR - o.aR * o.del;
        T lL, lR;
        interface_solve<T, S, SW, NWS, LS, Sh::P, LANES>(o.aL, DLr, ELr, FLr, ARr, DRr, o.cR, FRr,
                                                         tid, lane, sl, kw, ws, prm.iface,
                                                         prm.xchg_lds, tri_dyn_lds, lL, lR);
        lam[0] = lL;
        lam[M - 1] = lR;
        T ln = lR;
#pragma unroll
        for (int j = M - 3; j >= 0; --j) {
            ln = (o.de[j] - al_r[j] * lL) - o.ga[j] * ln;
            lam[j + 1] = ln;
        }
    }
    if constexpr (MODE == kAdjoint && kLater) take_last(rx, x_before, x_after);
    if (!IL && !valid) return;      // interleaved stores go by position, not by system

    // ------------------------------------------------------------ gradients
    // ga_i = -lambda_i x_{i-1}, gb_i = -lambda_i x_i, gc_i = -lambda_i x_{i+1}, gd_i = lambda_i
    auto grad = [&](int k, int j) -> T {
        const int64_t r = row0 + j;
        const T xm = (j == 0) ? x_before : rx[j - 1];
        const T xp = (j == M - 1) ? x_after : rx[j + 1];
        const T l = lam[j];
        if (k == 0) return (r > 0) ? -(l * xm) : T(0);
        if (k == 1) return -(l * rx[j]);
        if (k == 2) return (r < n - 1) ? -(l * xp) : T(0);
        if (k == 3) return l;
        return rx[j];
    };
    T *outs[5] = {prm.ga, prm.gb, prm.gc, prm.gd, prm.xo};
    constexpr int NOUT = (MODE == kFused) ? 5 : 4;
    if constexpr (IL) {
#pragma unroll
        for (int k = 0; k < NOUT; ++k) {
            T v[M];
#pragma unroll
            for (int j = 0; j < M; ++j) v[j] = grad(k, j);
            il_block_store<T, M, SW, S, NT, true>(make_rsrc(outs[k], prm.buf_bytes), wrow, prm.rstride,
                                                  (int64_t)tile * S, n, prm.batch, lane, sl, kw,
                                                  xbuf[wave], v);
        }
    } else {
        if (wrow >= n) return;                             // wave-uniform
#pragma unroll
        for (int k = 0; k < NOUT; ++k) {
            T v[M];
#pragma unroll
            for (int j = 0; j < M; ++j) v[j] = grad(k, j);
            adj_wave_store<T, M>(RW(outs[k]), wrow, lane, xbuf[wave], v);
        }
    }
}

template <typename T> struct AdjEntry {
    int M, NW, S;
    bool IL;
    int mode;
    int cap;
    hipError_t (*launch)(const AdjParams<T> &, hipStream_t);
};

template <typename T, int M, int NW, int S, bool IL, int MODE>
hipError_t launch_adj(const AdjParams<T> &p, hipStream_t st) {
    const int64_t tiles = (p.batch + S - 1) / S;
    if (tiles <= 0) return hipSuccess;
    if (tiles > 0x7fffffff) return hipErrorInvalidValue;
    // Interleaved: 128-byte pieces of rows on lines stream; narrower pieces and rows off
    // lines share lines with their neighbours, so the loads stay cached and runs of
    // neighbouring tiles go to one XCD.
    constexpr int LT = IL && S * (int)sizeof(T) < 128 ? 128 / (S * (int)sizeof(T)) : 1;
    const bool shared = IL && (LT > 1 || (p.rstride * (int64_t)sizeof(T)) % 128 != 0);
    AdjParams<T> q = p;
    q.line_tiles = shared && LT == 1 ? 16 : LT;
    auto kern = tile_adj_kernel<T, M, NW, S, IL, MODE, (LT == 1)>;
    if (shared) kern = tile_adj_kernel<T, M, NW, S, IL, MODE, !IL>;
    size_t dyn = 0;
    if (iface_family(p.iface) >= kIfacePCR) dyn = (size_t)iface_lds_bytes<T>(64 * NW);
    else if (p.xchg_lds) dyn = (size_t)6 * 64 * NW * sizeof(T);
    if (dyn) {
        static size_t granted[2] = {0, 0};
        if (dyn > granted[shared]) {
            hipFuncAttributes fa;
            hipError_t e = hipFuncGetAttributes(&fa, reinterpret_cast<const void *>(kern));
            if (e != hipSuccess) return e;
            if (fa.sharedSizeBytes + dyn > (size_t)max_lds_per_block()) return hipErrorInvalidConfiguration;
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn);
            if (e != hipSuccess) return e;
            granted[shared] = dyn;
        }
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(64 * NW), dyn, st, q);
    return hipGetLastError();
}

template <typename T> struct AdjTable {
    const AdjEntry<T> *entries;
    int count;
};
AdjTable<float> adj_table_f32();
AdjTable<double> adj_table_f64();
template <typename T> AdjTable<T> adj_table();
template <> inline AdjTable<float> adj_table<float>() { return adj_table_f32(); }
template <> inline AdjTable<double> adj_table<double>() { return adj_table_f64(); }

}  // namespace tri
