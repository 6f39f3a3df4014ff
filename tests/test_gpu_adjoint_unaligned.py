"""Adjoint and fused forward + adjoint of contiguous systems whose rows start at any
element: against the FP64 oracle, with the elements around every array untouched, and
with systems of NaN beside the checked ones (chunks at a system's end reach past it)."""
import ctypes

import numpy as np
import pytest

import oracle
from gpu_util import announce, make_case

pytestmark = pytest.mark.gpu

TOL = {np.float32: 1e-5, np.float64: 1e-12}


# around the tiles' capacities, the wave blocks (64 lanes of 4 or 8 rows) and the chunks
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 5, 255, 257, 383, 385, 511, 513, 767, 777, 1023, 1025, 1535, 1537, 2047,
                               3001, 3073, 4093, 4097, 6143, 6145])
@pytest.mark.parametrize("fused", [False, True])
def test_odd_rows(dtype, n, fused):
    import torch
    import tridiagonalsolver_amd as T
    batch, off, prec = 9, 1 + n % 3, int(dtype == np.float64)
    announce("adjoint unaligned", np.dtype(dtype).name, n, fused)
    a, b, c, d = make_case(n, batch, 0, dtype, seed=n)
    g = np.random.default_rng(n).standard_normal(n * batch).astype(dtype)
    x = oracle.thomas(a, b, c, d, n, batch)
    ref = [x] * fused + list(oracle.adjoint(a, b, c, x, g, n, batch))
    nan = np.arange(n * batch) // n % 2 == 1
    b = np.where(nan, np.nan, b).astype(dtype)
    ins = [a, b, c, d, g] if fused else [a, b, c, x.astype(dtype), g]
    m = n * batch

    def guarded(v):
        buf = torch.full((m + off + 37,), 7.0, dtype=torch.from_numpy(a).dtype, device="cuda")
        if v is not None:
            buf[off:off + m] = torch.from_numpy(v).cuda()
        return buf
    bufs = [guarded(v) for v in ins] + [guarded(None) for _ in ref]
    ptrs = [ctypes.c_void_p(t[off:].data_ptr()) for t in bufs]
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    fn = T.lib().tridiag_solve_fwd_bwd if fused else T.lib().tridiag_adjoint
    T.check(fn(prec, 0, n, batch, *ptrs, st))
    torch.cuda.synchronize()
    ends = torch.cat([torch.cat([t[:off], t[off + m:]]) for t in bufs])
    assert bool((ends == 7.0).all())
    for k, (t, r) in enumerate(zip(bufs[5:], ref)):
        o = t[off:off + m].cpu().numpy().astype(np.float64)[~nan]
        assert np.max(np.abs(o - r[~nan])) <= TOL[dtype] * max(np.max(np.abs(r)), 1e-300), k
