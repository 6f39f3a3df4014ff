"""Short contiguous systems, several per wave: every shape's capacity and the sizes beside
it, batches that leave the last wave and workgroup part empty, rows at any alignment,
against the FP64 oracle; the elements around the arrays stay untouched."""
import numpy as np
import pytest

from gpu_util import TOL, announce, check_against_oracle, make_case
from test_gpu_unaligned import solve_between_guards

pytestmark = pytest.mark.gpu

CAPS = [10, 14, 20, 28, 36, 40, 56, 72, 80, 112, 144, 160, 192]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("cap", CAPS)
def test_edges(dtype, cap):
    import tridiagonalsolver_amd as T
    prec = 0 if dtype == np.float32 else 1
    for n in sorted({9, cap - 1, cap, min(cap + 1, 192)}):
        for batch, off in ((1, 0), (65, 1), (131, 3), (1024, 0)):
            announce("short", np.dtype(dtype).name, n, batch, off)
            kind = "short" if n > 16 or batch > 64 else "lane"
            assert T.plan(prec, -1, 0, n, batch)["kind"] == kind
            arrs = make_case(n, batch, 0, dtype, seed=7 * n + batch)
            x, guards, same = solve_between_guards(arrs, n, batch, 0, -1, off)
            assert guards and same
            st, _ = check_against_oracle(arrs, x, n, batch, 0, dtype)
            assert st["nonfinite"] == 0 and st["relerr"] <= TOL[dtype], (n, batch, st)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_nan_stays_in_its_system(dtype):
    """Systems share a wave but not their values."""
    n, batch = 21, 200
    a, b, c, d = make_case(n, batch, 0, dtype, seed=3)
    b[5 * n + 2] = np.nan
    x, _, _ = solve_between_guards((a, b, c, d), n, batch, 0, -1, 0)
    bad = np.isnan(x.reshape(batch, n)).any(axis=1)
    assert bad[5] and bad.sum() == 1
