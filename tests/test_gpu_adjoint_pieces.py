"""Adjoint and fused forward + adjoint of interleaved systems on tiles that move whole row
pieces: sizes around the capacities, partial groups, rows on and off 128-byte lines, arrays at
any element; against the FP64 oracle, with the elements around every array untouched."""
import ctypes

import numpy as np
import pytest

import oracle
from gpu_util import announce, make_case

pytestmark = pytest.mark.gpu

TOL = {np.float32: 1e-5, np.float64: 1e-12}
CAPS = (16, 32, 48, 64, 96, 128, 192, 256, 384, 512, 768, 1024)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("fused", [False, True])
def test_any_size(dtype, fused):
    import torch
    import tridiagonalsolver_amd as T
    prec = int(dtype == np.float64)
    S = 16 if prec else 32
    fn = T.lib().tridiag_solve_fwd_bwd if fused else T.lib().tridiag_adjoint
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    fails = []
    for n in sorted({1, 2, 7} | {k + e for k in CAPS for e in (-1, 0, 1)}):
        for batch, off in ((1, 0), (S + 1, 1), (2 * S, 0)):
            announce("adjoint pieces", np.dtype(dtype).name, n, batch, fused)
            a, b, c, d = make_case(n, batch, 2, dtype, seed=n)
            g = np.random.default_rng(n).standard_normal(n * batch).astype(dtype)
            x = oracle.thomas(a, b, c, d, n, batch, layout=2)
            ref = [x] * fused + list(oracle.adjoint(a, b, c, x, g, n, batch, layout=2))
            m = n * batch

            def guarded(v):
                buf = torch.full((m + off + 37,), 7.0, dtype=torch.from_numpy(a).dtype, device="cuda")
                if v is not None:
                    buf[off:off + m] = torch.from_numpy(np.ascontiguousarray(v)).cuda()
                return buf
            ins = [a, b, c, d, g] if fused else [a, b, c, x.astype(dtype), g]
            bufs = [guarded(v) for v in ins] + [guarded(None) for _ in ref]
            T.check(fn(prec, 2, n, batch, *(ctypes.c_void_p(t[off:].data_ptr()) for t in bufs), st))
            ok = all(bool((t[:off] == 7).all() and (t[off + m:] == 7).all()) for t in bufs)
            errs = [np.max(np.abs(t[off:off + m].cpu().numpy().astype(np.float64) - r))
                    / max(np.max(np.abs(r)), 1e-300) for t, r in zip(bufs[5:], ref)]
            if not (ok and all(e <= TOL[dtype] for e in errs)):
                fails.append((n, batch, off, ok, errs))
    assert not fails, fails[:5]
