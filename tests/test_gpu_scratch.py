"""Scratch of the cooperative solve from the caller: exactly as much as is asked for, less
and none give the same bits as tridiag_solve, and the scratch's old contents do not matter."""
import ctypes

import pytest

from gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,layout,n,batch", [(0, 0, 20000, 7), (1, 0, 500000, 1),
                                                 (0, 2, 4096, 96), (1, 2, 2048, 40)])
def test_same_bits(prec, layout, n, batch):
    import torch
    import tridiagonalsolver_amd as T
    L = T.lib()
    dt = torch.float64 if prec else torch.float32
    a, c, d = (torch.rand(n * batch, device="cuda", dtype=dt) * 2 - 1 for _ in range(3))
    b = a.abs() + c.abs() + 1
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    need = L.tridiag_scratch_bytes(prec, -1, layout, n, batch)
    assert need > 0
    ref = d.clone()
    T.check(L.tridiag_solve(prec, -1, layout, n, batch, *(t.data_ptr() for t in (a, b, c, ref)),
                            stream))
    for size, fill in ((need, 0), (need, 255), (need // 2, 0), (0, 0)):
        announce("scratch", prec, layout, n, batch, size)
        w = torch.full((max(size, 1),), fill, device="cuda", dtype=torch.uint8)
        x = d.clone()
        for _ in range(2):                       # the second solve finds the first one's words
            x.copy_(d)
            T.check(L.tridiag_solve_scratch(prec, -1, layout, n, batch,
                                            *(t.data_ptr() for t in (a, b, c, x)),
                                            w.data_ptr() if size else None, size, stream))
            assert torch.equal(x, ref)
    assert L.tridiag_scratch_bytes(prec, -1, layout, 64, 3) == 0
