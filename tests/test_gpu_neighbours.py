"""Contiguous systems of any size beside systems and memory of NaN: chunks at a system's end
reach past it, so every array of the neighbours (not only the diagonal, which identity rows
replace) and the elements after the last system hold NaN.  The systems between them are
solved as if alone, against the FP64 oracle."""
import ctypes

import numpy as np
import pytest

import oracle
from gpu_util import TOL, announce, make_case

pytestmark = pytest.mark.gpu


def _between_nan(v, off):
    """v on the GPU from element `off` of a buffer that is NaN elsewhere."""
    import torch
    t = torch.from_numpy(v)
    buf = torch.full((off + v.size + 5000,), float("nan"), dtype=t.dtype, device="cuda")
    buf[off:off + v.size] = t.cuda()
    return buf[off:off + v.size]


def _every_other(arrs, n, batch):
    """NaN in all rows of the systems 1, 3, ...; returns the arrays and the rows to check."""
    bad = np.arange(n * batch) // n % 2 == 1
    return [np.where(bad, np.nan, v).astype(v.dtype) for v in arrs], ~bad


def _close(x, ref, dtype):
    return np.isfinite(x).all() and np.abs(x - ref).max() <= TOL[dtype] * np.abs(ref).max()


# several systems per wave, the tiles around their rows per lane and wave blocks, row blocks
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [11, 21, 55, 100, 190, 193, 300, 777, 1003, 2047, 3001, 5001, 8191,
                               20001, 70001])
def test_solve(dtype, n):
    import torch
    import tridiagonalsolver_amd as T
    batch = 65 if n < 5000 else 5
    announce("neighbours", np.dtype(dtype).name, n)
    arrs = make_case(n, batch, 0, dtype, seed=n)
    ref = oracle.thomas(*(v.astype(np.float64) for v in arrs), n, batch)
    nans, keep = _every_other(arrs, n, batch)
    ts = [_between_nan(v, 1) for v in nans]
    T.solve(*ts, n=n, batch=batch)
    torch.cuda.synchronize()
    assert _close(ts[3].cpu().numpy()[keep].astype(np.float64), ref[keep], dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_ragged(dtype):
    import torch
    import tridiagonalsolver_amd as T
    sizes = np.array([3, 17, 33, 65, 130, 257, 400, 700, 1001, 1500, 2049, 3000, 5001, 8191] * 5)
    off = oracle.offsets_from_sizes(sizes.astype(np.int64))
    announce("neighbours, ragged", np.dtype(dtype).name)
    arrs = [v.astype(dtype) for v in oracle.gen_dd_ragged(off, seed=5)]
    ref = oracle.thomas_ragged(*arrs, off)
    bad = np.repeat(np.arange(len(sizes)) % 2 == 1, sizes)
    ts = [_between_nan(np.where(bad, np.nan, v).astype(dtype), 1) for v in arrs]
    T.RaggedPlan(off, dtype=ts[0].dtype).solve(*ts)
    torch.cuda.synchronize()
    assert _close(ts[3].cpu().numpy()[~bad].astype(np.float64), ref[~bad], dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("n", [5, 100, 257, 385, 600, 777, 1025, 1400, 2047, 3001, 4093, 6001])
def test_adjoint(dtype, fused, n):
    import torch
    import tridiagonalsolver_amd as T
    batch = 9
    announce("neighbours, adjoint", np.dtype(dtype).name, n, fused)
    a, b, c, d = make_case(n, batch, 0, dtype, seed=n)
    g = np.random.default_rng(n).standard_normal(n * batch).astype(dtype)
    x = oracle.thomas(a, b, c, d, n, batch)
    ref = [x] * fused + list(oracle.adjoint(a, b, c, x, g, n, batch))
    nans, keep = _every_other([a, b, c, d if fused else x.astype(dtype), g], n, batch)
    ins = [_between_nan(v, 1) for v in nans]
    outs = [torch.empty(n * batch, dtype=ins[0].dtype, device="cuda") for _ in ref]
    fn = T.lib().tridiag_solve_fwd_bwd if fused else T.lib().tridiag_adjoint
    T.check(fn(int(dtype == np.float64), 0, n, batch,
               *(ctypes.c_void_p(t.data_ptr()) for t in ins + outs),
               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    for k, (t, r) in enumerate(zip(outs, ref)):
        assert _close(t.cpu().numpy()[keep].astype(np.float64), r[keep], dtype), k
