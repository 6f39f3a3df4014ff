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


@pytest.mark.parametrize("n,batch", [(3001, 40), (700, 33), (5000, 9)])
def test_captured_without_scratch(n, batch):
    """Interleaved sizes that the eager solve takes cooperatively, in a graph that is replayed
    on new values."""
    import torch
    import tridiagonalsolver_amd as T
    announce("captured solve", n, batch)
    a, c, d0 = (torch.rand(n, batch, device="cuda", dtype=torch.float64) * 2 - 1 for _ in range(3))
    b = a.abs() + c.abs() + 1
    d = d0.clone()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        T.solve(a, b, c, d, layout=2)                   # kernels are loaded
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        T.solve(a, b, c, d, layout=2)
    for k in range(4):
        rhs = d0 * (k + 1)
        d.copy_(rhs)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        T.solve(a, b, c, rhs, layout=2)
        assert float((d - rhs).abs().max()) <= 64 * 2.3e-16 * float(rhs.abs().max()), k


def test_two_streams():
    """Interleaved solves of several rounds on two streams at once."""
    import torch
    import tridiagonalsolver_amd as T
    n, batch = 1100, 4001
    vs = []
    for k in range(2):
        a, c, d = (torch.rand(n, batch, device="cuda") * 2 - 1 for _ in range(3))
        vs.append([a, a.abs() + c.abs() + 1, c, d])
    refs = [T.solve(*v[:3], v[3].clone(), layout=2) for v in vs]
    sts = [torch.cuda.Stream() for _ in vs]
    torch.cuda.synchronize()
    outs = [[], []]
    for i in range(4):
        for k, st in enumerate(sts):
            announce("two streams", i, k)
            with torch.cuda.stream(st):
                outs[k].append(T.solve(*vs[k][:3], vs[k][3].clone(), layout=2))
    torch.cuda.synchronize()
    for k in range(2):
        assert all(torch.equal(x, refs[k]) for x in outs[k])
