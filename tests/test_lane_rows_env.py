"""TRIDIAG_LANE_ROWS, the rows up to which the automatic choice takes one system per lane,
for every batch (the planner in a child process, without a GPU: the variable is read once)."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
import sys
sys.path.insert(0, %r)
import tridiagonalsolver_amd as T
print([T.plan(prec, -1, 0, n, batch)["kind"] for prec in (0, 1) for n in (8, 12, 16)
       for batch in (64, 65, 100000)])
"""


def kinds(rows):
    env = {k: v for k, v in os.environ.items() if k != "TRIDIAG_LANE_ROWS"}
    if rows is not None:
        env["TRIDIAG_LANE_ROWS"] = str(rows)
    r = subprocess.run([sys.executable, "-c", PROGRAM % ROOT], env=env, capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return eval(r.stdout)


def test_lane_rows():
    assert kinds(16) == ["lane"] * 18
    assert kinds(32) == ["lane"] * 18
    one = ["lane"] * 3 + ["lane"] * 3 + ["tile", "short", "short"]
    assert kinds(12) == one * 2
    default = ["lane"] * 3 + ["lane", "short", "short"] * 2
    assert kinds(None) == default * 2
