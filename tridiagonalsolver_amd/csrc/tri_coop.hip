// Cooperative row-block kernels: instantiations, launchers and their table.
#include <algorithm>
#include <mutex>

#include "tri_coop_tree.hpp"

namespace tri {

// Workgroups of 64 * NW lanes of `fn` that the current device holds at once (0 if
// unknown); cache[device] keeps the answer.
static int resident_workgroups(const void *fn, int lanes, int (&cache)[64]) {
    static std::mutex mu;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    std::lock_guard<std::mutex> lk(mu);
    int &c = cache[dev];
    if (c == 0) {
        int per_cu = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, lanes, 0) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        c = per_cu * cus;
    }
    return c;
}

// Interleaved systems.
template <typename T, int M, int NW, int S, int KMAX, int OCC>
static hipError_t launch_coop(const CoopParams<T> &p, int grid, hipStream_t st) {
    if (grid < 1 || p.K < 1 || p.K > KMAX || grid % p.K != 0) return hipErrorInvalidValue;
    if (p.pipelined)
        hipLaunchKernelGGL((coop_pipe_kernel<T, M, NW, S, KMAX>), dim3((unsigned)grid),
                           dim3(64 * NW), 0, st, p);
    else if (p.shared_lines)
        hipLaunchKernelGGL((coop_kernel<T, M, NW, S, KMAX, OCC, false>), dim3((unsigned)grid),
                           dim3(64 * NW), 0, st, p);
    else
        hipLaunchKernelGGL((coop_kernel<T, M, NW, S, KMAX, OCC, true>), dim3((unsigned)grid),
                           dim3(64 * NW), 0, st, p);
    return hipGetLastError();
}
template <typename T, int M, int NW, int S, int KMAX, int OCC>
static int coop_max_grid(bool pipelined) {
    static int cache[3][64];
    if (pipelined)
        return resident_workgroups(reinterpret_cast<const void *>(coop_pipe_kernel<T, M, NW, S, KMAX>),
                                   64 * NW, cache[2]);
    return std::min(
        resident_workgroups(reinterpret_cast<const void *>(coop_kernel<T, M, NW, S, KMAX, OCC, false>),
                            64 * NW, cache[0]),
        resident_workgroups(reinterpret_cast<const void *>(coop_kernel<T, M, NW, S, KMAX, OCC, true>),
                            64 * NW, cache[1]));
}

// Contiguous systems: the solve, and the pass over blocks whose wait gave up.
template <typename T, int M, int NW, int OCC>
static hipError_t launch_coop_tree(const CoopParams<T> &p, int grid, hipStream_t st) {
    if (grid < 1 || p.K < 1 || p.K > 64 * NW || grid % p.K != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL((coop_tree_kernel<T, M, NW, OCC>), dim3((unsigned)grid), dim3(64 * NW), 0,
                       st, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((coop_mend_kernel<T, M, NW, OCC>), dim3((unsigned)std::min(grid, 256)),
                       dim3(64 * NW), 0, st, p);
    return hipGetLastError();
}
template <typename T, int M, int NW, int OCC> static int coop_tree_max_grid(bool) {
    static int cache[64];
    return resident_workgroups(reinterpret_cast<const void *>(coop_tree_kernel<T, M, NW, OCC>),
                               64 * NW, cache);
}

__global__ void __launch_bounds__(256) coop_clear_kernel(uint64_t *w, int64_t count) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += (int64_t)gridDim.x * 256)
        w[i] = 0;
}
hipError_t launch_coop_clear(uint64_t *words, int64_t count, hipStream_t st) {
    hipLaunchKernelGGL(coop_clear_kernel, dim3((unsigned)std::min<int64_t>((count + 255) / 256, 256)),
                       dim3(256), 0, st, words, count);
    return hipGetLastError();
}

#define TRI_COOP_ENTRY(T, M, NW, S, KMAX, PIPE, OCC)                                          \
    {M, NW, S, true, CoopShape<T, M, NW, S>::R, KMAX, PIPE, &launch_coop<T, M, NW, S, KMAX, OCC>, \
     &coop_max_grid<T, M, NW, S, KMAX, OCC>}
#define TRI_COOP_TREE(T, M, NW, OCC)                                                          \
    {M, NW, 1, false, 64 * NW * M, 64 * NW, false, &launch_coop_tree<T, M, NW, OCC>,           \
     &coop_tree_max_grid<T, M, NW, OCC>}

// Interleaved: S systems = one 128-byte line per row, blocks of 2*NW*M (FP32) or
// 4*NW*M (FP64) rows, up to 64 blocks (16384 rows), two workgroups per CU.  PIPE:
// coop_pipe_kernel by default; OCC: waves per SIMD.  Measured on MI355X (us): pipelined
// instead FP32 4096 x 4096 100, FP64 211; blocks of 128 rows (M = 8 FP32, 4 FP64) and
// 16-wave workgroups were slower or even.
// With the block forms [system][block][6] in LDS (all lanes of an access on one bank), in a
// buffer of their own (one workgroup per CU above 32 blocks) and two serial chains, / now
// (back to back on the same arrays, scratch from the caller): FP32 4096 x 4096 81.1 / 80.2, 600 x
// 16,000 46.5 / 45.7, 8192 x 2048 108 / 106 (other placements of the arrays 85-97), 16,000 x 500
// 87.0 / 66.8; FP64 3001 x 1001 37.8 / 34.4, 3001 x 1008 32.1 / 27.1 (4.5 TB/s), 9000 x 250
// 54.1 / 42.0.  The loads' pattern alone (pieces of one line, 256 rows per task) takes 70-86
// us at FP32 4096 x 4096, which bounds the large sizes; the rest is the wait for the group
// and the phases that no second workgroup covers.
// Contiguous: one system, blocks of 64*NW*M rows, up to 64*NW blocks; small blocks
// first (choose_coop says which).  Both run 16 waves per CU, four or two workgroups.
static const CoopEntry<float> kCoopF32[] = {
    TRI_COOP_ENTRY(float, 16, 8, 32, 64, false, 4),
    TRI_COOP_TREE(float, 16, 4, 4),
    TRI_COOP_TREE(float, 16, 8, 4),
};
static const CoopEntry<double> kCoopF64[] = {
    TRI_COOP_ENTRY(double, 8, 8, 16, 64, false, 4),
    TRI_COOP_TREE(double, 8, 4, 4),
    TRI_COOP_TREE(double, 8, 8, 4),
};
#undef TRI_COOP_ENTRY
#undef TRI_COOP_TREE

CoopTable<float> coop_table_f32() { return {kCoopF32, (int)(sizeof(kCoopF32) / sizeof(kCoopF32[0]))}; }
CoopTable<double> coop_table_f64() {
    return {kCoopF64, (int)(sizeof(kCoopF64) / sizeof(kCoopF64[0]))};
}

}  // namespace tri
