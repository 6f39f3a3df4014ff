"""Contiguous systems whose rows are not 16-byte aligned (odd lengths, arrays that start
at any element) on the whole-chunk tiles: every solve against the FP64 oracle, and the
elements around the arrays untouched (chunks at a system's end reach past it)."""
import numpy as np
import pytest

import oracle
from gpu_util import TOL, announce, check_against_oracle, make_case

pytestmark = pytest.mark.gpu


def solve_between_guards(arrs, n, batch, layout, algo, off):
    """Solves copies that start `off` elements into larger buffers; returns x and the
    four buffers' elements before and after."""
    import torch
    import tridiagonalsolver_amd as T
    dev = torch.device("cuda:0")
    bufs, views = [], []
    for v in arrs:
        buf = torch.full((v.size + off + 37,), 7.0, dtype=torch.from_numpy(v).dtype, device=dev)
        buf[off:off + v.size] = torch.from_numpy(v).to(dev)
        bufs.append(buf)
        views.append(buf[off:off + v.size])
    if layout == 1:
        T.solve(views[0], None, None, None, algo=algo, layout=1, n=n, batch=batch)
    else:
        T.solve(*views, algo=algo, layout=layout, n=n, batch=batch)
    torch.cuda.synchronize()
    x = views[0 if layout == 1 else 3].cpu().numpy()
    ends = torch.cat([torch.cat([b[:off], b[off + v.size:]]) for b, v in zip(bufs, arrs)])
    same = all(bool(torch.equal(views[k].cpu(), torch.from_numpy(arrs[k]))) for k in range(3)) \
        if layout != 1 else True
    return x, bool((ends == 7.0).all()), same


# one chunk and one row around the tiles' capacities, rows per lane and wave blocks
SIZES = [193, 255, 257, 385, 511, 767, 1001, 1023, 1537, 2047, 3071, 4095, 5001, 8191]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", SIZES)
def test_odd_rows(dtype, n):
    batch = 11
    for layout, algo, off in ((0, -1, 0), (0, -1, 3), (0, 5, 1), (1, 9, 1)):
        announce("unaligned", np.dtype(dtype).name, n, layout, algo, off)
        arrs = make_case(n, batch, layout, dtype, seed=n + off)
        x, guards, same = solve_between_guards(arrs, n, batch, layout, algo, off)
        assert guards and same
        st, _ = check_against_oracle(arrs, x, n, batch, layout, dtype)
        assert st["relerr"] <= TOL[dtype], (n, layout, algo, off, st)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_neighbours_are_not_read(dtype):
    """A system's result does not depend on the systems beside it (NaN in every other
    system stays there)."""
    n, batch = 1003, 8
    a, b, c, d = make_case(n, batch, 0, dtype, seed=5)
    ref = oracle.thomas(*(v.astype(np.float64) for v in (a, b, c, d)), n, batch)
    for s in range(1, batch, 2):
        b[s * n:(s + 1) * n] = np.nan
    x, guards, _ = solve_between_guards((a, b, c, d), n, batch, 0, -1, 1)
    assert guards
    x, ref = x.reshape(batch, n)[::2], ref.reshape(batch, n)[::2]
    assert np.linalg.norm(x - ref) <= TOL[dtype] * np.linalg.norm(ref)
