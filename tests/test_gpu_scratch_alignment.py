"""Scratch from the caller that is not aligned to 8 bytes, which the kernels' 64-bit words
need, is left alone: the solve allocates, with the bits of the aligned one."""
import ctypes

import pytest

from gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,layout,n,batch", [(0, 0, 20000, 7), (1, 0, 70000, 3), (0, 2, 4096, 96),
                                                 (1, 2, 3001, 40)])
@pytest.mark.parametrize("off", [0, 1, 4, 8])
def test_misaligned(prec, layout, n, batch, off):
    import torch
    import tridiagonalsolver_amd as T
    L = T.lib()
    announce("scratch alignment", prec, layout, n, batch, off)
    dt = torch.float64 if prec else torch.float32
    a, c, d = (torch.rand(n * batch, device="cuda", dtype=dt) * 2 - 1 for _ in range(3))
    b = a.abs() + c.abs() + 1
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ref = d.clone()
    T.check(L.tridiag_solve(prec, -1, layout, n, batch, *(t.data_ptr() for t in (a, b, c, ref)),
                            stream))
    need = L.tridiag_scratch_bytes(prec, -1, layout, n, batch)
    w = torch.full((need + off,), 171, device="cuda", dtype=torch.uint8)
    T.check(L.tridiag_solve_scratch(prec, -1, layout, n, batch, *(t.data_ptr() for t in (a, b, c, d)),
                                    w.data_ptr() + off, need, stream))
    torch.cuda.synchronize()
    assert torch.equal(d, ref)
    assert bool((w == 171).all()) == (off % 8 != 0)
