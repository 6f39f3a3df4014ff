"""Short contiguous systems (up to 32 FP32 / 16 FP64 rows) with a zero or tiny diagonal entry
whose Thomas pivots are all of order one: the automatic choice solves them by the Thomas
recurrence at any batch, with the bits of the Thomas id.

a, c ~ U[0.5, 1], b ~ U[4, 5] but for one row per system, where b is 0 or +-1e-9: c' stays in
[0.1, 0.3] up to that row, its pivot in [-0.3, -0.05], c' there in [-20, -1], and the next
pivot is above 4.  One pivot grows the error by at most 20, so |error| <= 20 * 64 eps max|x|
(64 eps as for dominant systems)."""
import numpy as np
import pytest

import oracle
from gpu_util import announce, run_solve

pytestmark = pytest.mark.gpu


def _systems(n, batch, dtype, seed):
    rng = np.random.default_rng(seed)
    a, c = rng.uniform(0.5, 1.0, (2, batch, n))
    b = rng.uniform(4.0, 5.0, (batch, n))
    s = np.arange(batch)
    b[s, 1 + s % (n - 1)] = np.array([0.0, 1e-9, -1e-9])[s // (n - 1) % 3]
    d = rng.uniform(-1.0, 1.0, (batch, n))
    return tuple(np.ascontiguousarray(v.ravel().astype(dtype)) for v in (a, b, c, d))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_thomas_pivots(dtype):
    for n in range(2, (32 if dtype == np.float32 else 16) + 1):
        for batch in (64, 65, 131, 1000):
            announce("short pivots", np.dtype(dtype).name, n, batch)
            arrs = _systems(n, batch, dtype, n * 1000 + batch)
            x = run_solve(arrs, n, batch, 0, -1, dtype)
            ref = oracle.thomas(*(v.astype(np.float64) for v in arrs), n, batch)
            err = np.abs(x - ref).max()
            assert err <= 20 * 64 * np.finfo(dtype).eps * np.abs(ref).max(), (n, batch, err)
            assert np.array_equal(x, run_solve(arrs, n, batch, 0, 1, dtype)), (n, batch)
