// Which group of systems a slot of the cooperative schedule solves.  Plain C++
// shared by the kernels and the host checks.
#pragma once

#if defined(__HIPCC__)
#define TRI_COOP_HD __host__ __device__
#else
#define TRI_COOP_HD
#endif

namespace tri {

// Group solved by slot s (tasks s*K .. s*K + K-1) of G groups.  A round of the
// persistent grid runs W = P/K slots at once.  With W > 1, the W slots of a round
// take groups R = ceil(G/W) apart: slot s = r*W + c is entry (row r, column c) of a
// column-major table of W columns, the first L = G - (R-1)*W of which hold R
// entries and the rest R - 1.  A round's loads then cover the whole width of an
// interleaved row instead of a strip of W*S neighbouring systems.  Measured with
// the kernels' own load pattern at FP32 4096 x 4096 (128-byte row pieces, 32
// groups per round): 3.2 TB/s with neighbouring groups, 3.9 TB/s spread.  The map
// is a bijection on [0, G) for every W; which slots share a round is unchanged,
// so every wait of the schedule still ends.
inline TRI_COOP_HD int coop_group(int s, int G, int W) {
    if (W <= 1 || G <= W) return s;
    const int R = (G + W - 1) / W;
    const int r = s / W, c = s - r * W;
    const int L = G - (R - 1) * W;
    return c < L ? c * R + r : L * R + (c - L) * (R - 1) + r;
}

// Group gi and row block j of task `task` of a grid of P workgroups (P a multiple of K)
// when the row pieces of neighbouring groups share lines.  A round's groups are neighbours
// and come in clusters of C whose tasks are consecutive; a cluster's tasks are numbered row
// block by row block, and each XCD (workgroups are dispatched to the eight in turn) takes
// consecutive numbers, so that its L2 serves the second reader of a line.  C * K stays
// at most 64, what a system of 64 blocks needs by itself, so that few workgroups wait for
// each other where some of the grid cannot run.
// Measured on MI355X, C * K <= 128 / <= 64 (us): FP64 3001 x 1001 40.4 / 39.9, 1024 x 4001
// 53.9 / 55.5, 9000 x 250 41.7 / 43.2, FP32 4096 x 4001 103.5 / 103.5, 600 x 15,999 66.0 / 64.0.
inline TRI_COOP_HD void coop_task_shared(int task, int P, int K, int G, int &gi, int &j) {
    const int C = K <= 16 ? 4 : K <= 32 ? 2 : 1;
    const int round = task / P, b = task - round * P;
    const int first = round * (P / K), W = G - first < P / K ? G - first : P / K;
    const int cl = b / (C * K), c = b - cl * (C * K);
    const int w = W - cl * C < C ? W - cl * C : C;          // groups of this cluster
    const int active = w * K, q = active / 8, r = active % 8, x = c % 8;
    const int pos = x * q + (x < r ? x : r) + c / 8;
    j = pos / w;
    gi = first + cl * C + pos - j * w;
}

}  // namespace tri
