"""The cooperative schedule of interleaved rows off 128-byte lines (coop_task_shared, plain
C++), on the host: the K tasks of a group lie in one round of the grid and within 64
consecutive workgroups (a cluster of groups holds at most 64 tasks)."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "tridiagonalsolver_amd", "csrc")

PROGRAM = r"""
#include "tri_coop_sched.hpp"
#include <cstdio>
#include <vector>
int main() {
    for (int K = 1; K <= 64; ++K)
        for (int cap : {K, 96, 250, 256, 511, 512})
            for (int G : {1, 2, 3, 7, 8, 9, 31, 32, 33, 64, 65, 100, 257}) {
                if (cap < K) continue;
                const int P = cap / K * K < G * K ? cap / K * K : G * K;
                std::vector<int> lo(G, -1), hi(G, -1);
                for (int t = 0; t < G * K; ++t) {
                    int g, j;
                    tri::coop_task_shared(t, P, K, G, g, j);
                    if (g < 0 || g >= G) return 1;
                    if (lo[g] < 0) lo[g] = t;
                    hi[g] = t;
                }
                for (int g = 0; g < G; ++g)
                    if (lo[g] / P != hi[g] / P || hi[g] - lo[g] >= 64) return 2;
            }
    std::puts("ok");
    return 0;
}
"""


def test_span(tmp_path):
    src, exe = tmp_path / "sched.cpp", tmp_path / "sched"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True).stdout == "ok\n"
