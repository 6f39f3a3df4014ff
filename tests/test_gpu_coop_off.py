"""The routes of long systems without the cooperative solve (TRIDIAG_COOP_MIN_ROWS=-1 in a
child process; a captured interleaved solve without scratch takes them too): interleaved
tiles above 512 rows, on and off 128-byte lines, the contiguous copy above 4096 rows, and
the chunked contiguous solve, against the FP64 oracle."""
import os
import subprocess
import sys

import pytest

from gpu_util import announce

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
import sys, numpy as np
sys.path.insert(0, %(root)r)
sys.path.insert(0, %(root)r + '/tests')
import tridiagonalsolver_amd as T
from gpu_util import TOL, announce, check_against_oracle, make_case, run_solve
for layout, n, batch, kind in (
        (2, 513, 33, "tile"), (2, 600, 96, "tile"), (2, 767, 1, "tile"), (2, 768, 64, "tile"),
        (2, 1001, 40, "tile"), (2, 1024, 64, "tile"), (2, 2048, 17, "tile"), (2, 2100, 64, "tile"),
        (2, 3001, 40, "tile"), (2, 4096, 64, "tile"), (2, 4096, 4001, "tile"),
        (2, 4097, 9, "via_contiguous"), (2, 5000, 64, "via_contiguous"), (2, 8191, 20, "via_contiguous"),
        (2, 16384, 21, "via_contiguous"), (0, 20001, 7, "chunked"), (0, 131073, 3, "chunked"),
        (0, 300000, 2, "chunked")):
    for dtype in (np.float32, np.float64):
        announce("cooperative off", np.dtype(dtype).name, layout, n, batch)
        p = T.plan(int(dtype == np.float64), -1, layout, n, batch)
        assert p["kind"] == kind and "K" not in p, p
        arrs = make_case(n, batch, layout, dtype, seed=n + batch)
        x = run_solve(arrs, n, batch, layout, -1, dtype)
        st, _ = check_against_oracle(arrs, x, n, batch, layout, dtype)
        assert st["nonfinite"] == 0 and st["relerr"] <= TOL[dtype], st
print("ok", flush=True)
"""


def test_routes_without_it():
    announce("cooperative solve off (child process)")
    r = subprocess.run([sys.executable, "-c", PROGRAM % {"root": ROOT}],
                       env=dict(os.environ, TRIDIAG_COOP_MIN_ROWS="-1"), capture_output=True,
                       text=True, timeout=110)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
