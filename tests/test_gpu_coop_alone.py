"""Interleaved cooperative solves whose waits give up: with TRIDIAG_COOP_SPIN=0 a wait gives up
unless every other block of the group is there at its first look, which is what happens
where workgroups of the grid cannot run beside each other.  The workgroup then reduces the
missing blocks itself: x has the bits of the undisturbed solve everywhere, in place and in
an array of its own, in both cooperative kernels, and under replays of a captured solve."""
import os
import subprocess
import sys

import numpy as np
import pytest

from gpu_util import announce

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# partial blocks and groups, rows on and off lines, 3 to 64 blocks, one round and several
CASES = [(0, 600, 33), (0, 513, 20001), (0, 4096, 4096), (0, 3001, 4001), (0, 16384, 96),
         (0, 9001, 777), (1, 5000, 9), (1, 3001, 1001), (1, 4096, 2048), (1, 16129, 48)]

PROGRAM = r"""
import sys, numpy as np, torch
sys.path.insert(0, %(root)r)
import tridiagonalsolver_amd as T
out = {}
for i, (prec, n, batch) in enumerate(%(cases)r):
    dt = torch.float64 if prec else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(i)
    a, c, d = (torch.rand(n, batch, generator=gen, device="cuda", dtype=dt) * 2 - 1 for _ in range(3))
    b = a.abs() + c.abs() + 1
    assert T.plan(prec, -1, 2, n, batch)["K"] > 1
    print("[gpu-case]", prec, n, batch, flush=True)
    x = T.tridiagonal_solve(a, b, c, d, layout=2)
    if n * batch < 4000000:
        g, e, st = torch.cuda.CUDAGraph(), d.clone(), torch.cuda.Stream()
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(st):
            T.solve(a, b, c, e, layout=2)
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=st):
            T.solve(a, b, c, e, layout=2)
        for k in range(3):
            e.copy_(d)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            out["replay%%d_%%d" %% (i, k)] = e.cpu().numpy()
    T.solve(a, b, c, d, layout=2)
    out["x%%d" %% i], out["to%%d" %% i] = d.cpu().numpy(), x.cpu().numpy()
np.savez(%(path)r, **out)
print("ok", flush=True)
"""


def _run(path, env):
    announce("waits give up (child process)", env)
    r = subprocess.run([sys.executable, "-c", PROGRAM % {"root": ROOT, "cases": CASES, "path": path}],
                       env=dict(os.environ, **env), capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
    return np.load(path)


@pytest.mark.parametrize("pipe", ["0", "1"])
def test_waits_that_give_up(tmp_path, pipe):
    ref = _run(str(tmp_path / "ref.npz"), {"TRIDIAG_COOP_PIPE": pipe})
    got = _run(str(tmp_path / "got.npz"), {"TRIDIAG_COOP_PIPE": pipe, "TRIDIAG_COOP_SPIN": "0"})
    assert sorted(ref.files) == sorted(got.files)
    for k in ref.files:
        assert np.isfinite(ref[k]).all() and np.array_equal(got[k], ref[k]), k
