"""Long contiguous systems solved by up to 512 workgroups each (coop_tree_kernel), against
the FP64 oracle: block counts at the edges of the waves' 64-block groups and of the two
block sizes, several rounds of the grid, waits that give up, overlapping solves on two
streams, and replays of a captured solve."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from gpu_util import TOL, announce, check_against_oracle, make_case, run_solve

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("dtype,n,batch", [
    # FP32: blocks of 4096 rows (33, 64, 65, 129, 256 of them), then of 8192
    (np.float32, 131073, 5), (np.float32, 262144, 3), (np.float32, 262145, 2),
    (np.float32, 4096 * 128 + 1, 1), (np.float32, 1 << 20, 1), (np.float32, (1 << 20) + 3, 1),
    (np.float32, 270001, 40), (np.float32, 540001, 9), (np.float32, 1 << 22, 1),
    (np.float32, (1 << 22) + 1, 1),
    # FP64: 2048 rows, then 4096
    (np.float64, 65537, 5), (np.float64, 131072, 3), (np.float64, 131073, 2),
    (np.float64, 524288, 1), (np.float64, 524289, 1), (np.float64, 135001, 40),
    (np.float64, 700000, 4), (np.float64, 1 << 21, 1), (np.float64, (1 << 21) + 1, 1)])
def test_against_oracle(dtype, n, batch):
    announce("long systems", np.dtype(dtype).name, n, batch)
    arrs = make_case(n, batch, 0, dtype, seed=n % 997 + batch, blo=0.05, bhi=0.2)
    x = run_solve(arrs, n, batch, 0, -1, dtype)
    st, _ = check_against_oracle(arrs, x, n, batch, 0, dtype)
    assert st["nonfinite"] == 0 and st["relerr"] <= TOL[dtype], st


_GIVE_UP = r"""
import sys, numpy as np
sys.path.insert(0, %(root)r)
sys.path.insert(0, %(root)r + '/tests')
from gpu_util import TOL, check_against_oracle, make_case, run_solve
for dtype, n, batch in ((np.float32, 20001, 300), (np.float32, 300000, 20), (np.float64, 70001, 40),
                        (np.float64, 600000, 3)):
    arrs = make_case(n, batch, 0, dtype, seed=n)
    x = run_solve(arrs, n, batch, 0, -1, dtype)
    st, _ = check_against_oracle(arrs, x, n, batch, 0, dtype)
    print(np.dtype(dtype).name, n, st['relerr'], flush=True)
    assert st['nonfinite'] == 0 and st['relerr'] <= TOL[dtype], st
print('ok', flush=True)
"""


def test_waits_that_give_up():
    """TRIDIAG_COOP_SPIN=0: a wait gives up unless every block is there at its first
    look; the second pass solves those blocks and x is right everywhere."""
    announce("long systems, waits give up (child process)")
    r = subprocess.run([sys.executable, "-c", _GIVE_UP % {"root": ROOT}],
                       env=dict(os.environ, TRIDIAG_COOP_SPIN="0"), capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_two_streams(dtype):
    """Two streams solve at the same time; neither keeps the other from its answer."""
    import torch
    import tridiagonalsolver_amd as T
    n, batch = 1 << 20, 4
    announce("long systems on two streams", np.dtype(dtype).name)
    cases = []
    for k in range(2):
        arrs = make_case(n, batch, 0, dtype, seed=k)
        ref = oracle.thomas(*(v.astype(np.float64) for v in arrs), n, batch)
        cases.append(([torch.from_numpy(v).cuda().view(batch, n) for v in arrs], ref,
                      torch.cuda.Stream()))
    torch.cuda.synchronize()
    xs = [[], []]
    for _ in range(4):
        for k, (v, _, st) in enumerate(cases):
            with torch.cuda.stream(st):
                x = v[3].clone()
                T.solve(v[0], v[1], v[2], x)
                xs[k].append(x)
    torch.cuda.synchronize()
    for k, (_, ref, _) in enumerate(cases):
        for x in xs[k]:
            e = np.abs(x.cpu().numpy().ravel().astype(np.float64) - ref).max()
            assert e <= TOL[dtype] * np.abs(ref).max()


@pytest.mark.parametrize("layout,n,batch", [(0, 300000, 3), (0, 20000, 7), (2, 4096, 64)])
def test_captured_solve_replays(layout, n, batch):
    """Every replay of a captured solve solves what the arrays hold then."""
    import torch
    import tridiagonalsolver_amd as T
    announce("captured cooperative solve", layout, n)
    bufs = [torch.empty(n * batch, device="cuda") for _ in range(4)]
    st = torch.cuda.Stream()

    def call():
        T.check(T.lib().tridiag_solve_noalloc(0, -1, layout, n, batch,
                                              *(ctypes.c_void_p(t.data_ptr()) for t in bufs),
                                              ctypes.c_void_p(st.cuda_stream)))

    def fill(seed):
        arrs = make_case(n, batch, layout, np.float32, seed=seed)
        for t, v in zip(bufs, arrs):
            t.copy_(torch.from_numpy(v))
        torch.cuda.synchronize()
        return arrs
    fill(0)
    with torch.cuda.stream(st):
        call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        call()
    for seed in range(1, 5):
        arrs = fill(seed)
        g.replay()
        torch.cuda.synchronize()
        x = bufs[3].cpu().numpy()
        ref = oracle.thomas(*(v.astype(np.float64) for v in arrs), n, batch, layout=layout)
        assert np.abs(x - ref).max() <= TOL[np.float32] * np.abs(ref).max(), seed
