// Short contiguous systems: P lanes per system, 64/P systems per wave, M rows per
// lane, on chip (5 words of HBM traffic per unknown).
//
// The systems of a wave are consecutive, so their rows are one block of 64/P * n
// elements per array.  The wave reads it as whole 16-byte chunks (consecutive lanes,
// consecutive chunks, whatever the block's alignment: the buffer checks each dword
// against the block's end), hands the rows to the lanes through its LDS block, sweeps
// each lane's rows and merges the P segments of every system in log2(P) Wang-Mou
// rounds; the merged block is the system, so x of each segment's ends is its r.  No
// workgroup barrier, no chain over wave blocks.
//
// Up to the rows that one lane holds (32 FP32, 16 FP64) the systems are solved by the Thomas
// recurrence across their lanes instead (thomas_rows), operation by operation as the lane
// kernel does: the segments' elimination starts at their second row, so it fails or loses
// digits where a diagonal entry there is zero or small, which the Thomas pivots need not be.
// Segments / Thomas at 2^22 unknowns, back to back (us): FP32 9 rows 12.7 / 12.7, 16 rows 14.3 /
// 14.6, 28 rows 13.7 / 14.1; FP64 9 rows 26.3 / 26.4, 16 rows 27.2 / 27.8.
//
// What bounds it: memory, once the lanes hold rows.  The one-workgroup tiles give a
// system at least a whole wave, so that below 64 rows per 2-row segment most lanes
// held padding, and read their rows one element at a time.  M is odd: a lane's rows
// start M elements after its neighbour's, and an odd stride puts the 64 reads of a
// row on distinct LDS banks.
// Measured on MI355X at 2^22 unknowns (us, kernel before -> this): FP32 9 rows 21.1 ->
// 14.7, 17 rows 32.1 -> 15.3, 33 rows 50.4 -> 16.6, 64 rows 27.3 -> 15.0, 100 rows 20.6
// -> 16.4; FP64 9 rows 42.1 -> 28.2, 17 rows 183 -> 28.2 (5.9 TB/s), 33 rows 97.5 ->
// 29.1, 64 rows 55.6 -> 28.2, 100 rows 39.7 -> 29.9.
#include "tri_host.hpp"

namespace tri {

template <typename T, int M> struct ShortShape {
    static constexpr int M_ = M, NI = M - 2;
    static constexpr int CH = M, NC = 1, NBUF = 1;   // rows are in registers already
};

// x of the lane's rows (the first is the system's row row0 of nr; identity rows past it) by the
// Thomas recurrence over the P lanes of every system.  A lane's sweep starts from its
// neighbour's last row; all lanes sweep in every round, and after round t the first t + 1
// lanes of a system hold their final rows (P <= 4: what the others compute costs less than
// branches around it).
template <typename T, int M, int P>
__device__ __forceinline__ void thomas_rows(const T (&rows)[4][M], int row0, int nr, int lane,
                                            T (&xs)[M]) {
    const bool first = lane % P == 0, last = lane % P == P - 1;
    T cq[M], dq[M];
#pragma unroll
    for (int t = 0; t < P; ++t) {
        T cp = 0, dp = 0;
        if (t > 0) {
            cp = lane_read(cq[M - 1], lane - 1);
            dp = lane_read(dq[M - 1], lane - 1);
            if (first) { cp = 0; dp = 0; }
        }
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const T aj = (row0 + j == 0) ? T(0) : rows[0][j];        // a_0 is not part of A
            const T cj = (row0 + j == nr - 1) ? T(0) : rows[2][j];   // nor is c_{n-1}
            const T k = rcp(rows[1][j] - aj * cp);
            cp = cj * k;
            dp = (rows[3][j] - aj * dp) * k;
            cq[j] = cp;
            dq[j] = dp;
        }
    }
#pragma unroll
    for (int t = 0; t < P; ++t) {
        T xn = 0;
        if (t > 0) {
            xn = lane_read(xs[0], lane + 1);
            if (last) xn = 0;
        }
#pragma unroll
        for (int j = M - 1; j >= 0; --j) {
            xn = dq[j] - cq[j] * xn;
            xs[j] = xn;
        }
    }
}

template <typename T, int M, int P, bool THOMAS>
__global__ void __launch_bounds__(256) short_kernel(const T *a, const T *b, const T *c,
                                                    const T *d, T *x, int64_t n, int64_t batch) {
    using Sh = ShortShape<T, M>;
    constexpr int G = 64 / P;                            // systems per wave
    constexpr int TOT = 64 * M * (int)sizeof(T) / 16;    // 16-byte chunks of a full block
    constexpr int NQ = (TOT + 63) / 64;                  // chunk loads per lane
    __shared__ u32x4 lds[4][TOT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t sys0 = ((int64_t)blockIdx.x * 4 + wave) * G;   // first system of the wave
    if (sys0 >= batch) return;                                   // wave-uniform, no barriers
    const int nr = (int)n;
    const int64_t nsw = (batch - sys0 < G) ? batch - sys0 : G;
    const int32_t nb = (int32_t)(nsw * n * (int64_t)sizeof(T));
    const int64_t base = wave_uniform(sys0 * n);
    const __amdgpu_buffer_rsrc_t rr[4] = {make_rsrc(a + base, nb), make_rsrc(b + base, nb),
                                          make_rsrc(c + base, nb), make_rsrc(d + base, nb)};
    u32x4 *xb = lds[wave];
    T *tb = reinterpret_cast<T *>(xb);
    u32x4 g[4][NQ];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            g[k][q] = load16<true>(rr[k], lane * 16 + q * 1024);
    const int row0 = (lane % P) * M;                  // the lane's first row
    const int e0 = (lane / P) * nr + row0;            // its element of the block
    T rows[4][M];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (k > 0) wave_lds_sync();
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            if ((q + 1) * 64 <= TOT || q * 64 + lane < TOT) xb[q * 64 + lane] = g[k][q];
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < M; ++j) {
            // e0 + j < 64 * M: the block's (G - 1) * n + P * M at most.  Rows past the
            // system are identity rows; in the systems past the batch n rows of zeros
            // come from the buffer's bounds and are replaced like them
            const T v = tb[e0 + j];
            rows[k][j] = (row0 + j < nr) ? v : T(k == 1 ? 1 : 0);
        }
    }
    if constexpr (THOMAS) {
        T xs[M];
        thomas_rows<T, M, P>(rows, row0, nr, lane, xs);
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < M; ++j)
            if (row0 + j < nr) tb[e0 + j] = xs[j];
    } else {
        T al[Sh::NI];
        SweepOut<T, Sh::NI> o;
        RegLoader<T, M, M> ld{rows};
        lane_sweep<T, Sh>(o, ld, row0, n, [&](int j, T v) { al[j] = v; });
        const T DLr = o.bL - o.cL * o.SA, ELr = o.cL * o.PI, FLr = o.dL - o.cL * o.SD;
        const T ARr = -(o.aR * o.alp), DRr = o.bR - o.aR * o.g, FRr = o.dR - o.aR * o.del;
        Outer<T> oL, oR;
        segment_outer(o.aL, DLr, ELr, FLr, ARr, DRr, o.cR, FRr, oL, oR);
        wm_wave_merges<T, P, 1>(oL, oR, lane, 0, lane, P, false, nullptr);
        T xn = oR.r;
        wave_lds_sync();
        if (row0 + M - 1 < nr) tb[e0 + M - 1] = xn;
#pragma unroll
        for (int j = M - 3; j >= 0; --j) {
            xn = (o.de[j] - al[j] * oL.r) - o.ga[j] * xn;
            if (row0 + j + 1 < nr) tb[e0 + j + 1] = xn;
        }
        if (row0 < nr) tb[e0] = oL.r;
    }
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < NQ; ++q)
        if ((q + 1) * 64 <= TOT || q * 64 + lane < TOT)
            store16<true>(xb[q * 64 + lane], make_rsrc(x + base, nb), lane * 16 + q * 1024);
}

template <typename T, int M, int P, bool THOMAS>
static hipError_t launch_short_shape(const T *a, const T *b, const T *c, const T *d, T *x,
                                     int64_t n, int64_t batch, hipStream_t st) {
    constexpr int G = 64 / P;
    const int64_t blocks = (batch + 4 * G - 1) / (4 * G);
    if (n > P * M || blocks > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((short_kernel<T, M, P, THOMAS>), dim3((unsigned)blocks), dim3(256), 0, st, a,
                       b, c, d, x, n, batch);
    return hipGetLastError();
}

// Shapes by capacity P * M; the smallest that holds n runs.
template <typename T> struct ShortEntry {
    int M, P;
    hipError_t (*launch)(const T *, const T *, const T *, const T *, T *, int64_t, int64_t,
                         hipStream_t);
};
#define TRI_SHORT(T, M, P) {M, P, &launch_short_shape<T, M, P, false>}
#define TRI_SHORT_TABLE(T) \
    TRI_SHORT(T, 5, 2), TRI_SHORT(T, 7, 2), TRI_SHORT(T, 5, 4), \
    TRI_SHORT(T, 7, 4), TRI_SHORT(T, 9, 4), TRI_SHORT(T, 5, 8), TRI_SHORT(T, 7, 8), \
    TRI_SHORT(T, 9, 8), TRI_SHORT(T, 5, 16), TRI_SHORT(T, 7, 16), TRI_SHORT(T, 9, 16), \
    TRI_SHORT(T, 5, 32), TRI_SHORT(T, 7, 32)
static const ShortEntry<float> kShortF32[] = {TRI_SHORT_TABLE(float)};
static const ShortEntry<double> kShortF64[] = {TRI_SHORT_TABLE(double)};
#undef TRI_SHORT_TABLE
#undef TRI_SHORT
// By the Thomas recurrence: up to the rows of the lane kernel.
#define TRI_SHORT_THOMAS(T, M, P) {M, P, &launch_short_shape<T, M, P, true>}
static const ShortEntry<float> kThomasF32[] = {
    TRI_SHORT_THOMAS(float, 5, 2), TRI_SHORT_THOMAS(float, 7, 2), TRI_SHORT_THOMAS(float, 5, 4),
    TRI_SHORT_THOMAS(float, 7, 4), TRI_SHORT_THOMAS(float, 9, 4)};
static const ShortEntry<double> kThomasF64[] = {
    TRI_SHORT_THOMAS(double, 5, 2), TRI_SHORT_THOMAS(double, 7, 2), TRI_SHORT_THOMAS(double, 5, 4)};
#undef TRI_SHORT_THOMAS

template <typename T, int N>
static hipError_t launch_short(const ShortEntry<T> (&tab)[N], const T *a, const T *b, const T *c,
                               const T *d, T *x, int64_t n, int64_t batch, hipStream_t st) {
    if (batch <= 0) return hipSuccess;
    for (const ShortEntry<T> &e : tab)
        if (n <= e.M * e.P) return e.launch(a, b, c, d, x, n, batch, st);
    return hipErrorInvalidValue;
}

hipError_t launch_short_f32(const float *a, const float *b, const float *c, const float *d, float *x,
                            int64_t n, int64_t batch, bool thomas, hipStream_t st) {
    return thomas ? launch_short(kThomasF32, a, b, c, d, x, n, batch, st)
                  : launch_short(kShortF32, a, b, c, d, x, n, batch, st);
}
hipError_t launch_short_f64(const double *a, const double *b, const double *c, const double *d,
                            double *x, int64_t n, int64_t batch, bool thomas, hipStream_t st) {
    return thomas ? launch_short(kThomasF64, a, b, c, d, x, n, batch, st)
                  : launch_short(kShortF64, a, b, c, d, x, n, batch, st);
}

}  // namespace tri
