"""tridiag_solve_to: x in an array of its own has the bits of the solve in place, the inputs
are only read (c aside, for the Thomas id) and nothing around x is written; one shape of every
path, with arrays at any element."""
import ctypes

import pytest

from gpu_util import announce

pytestmark = pytest.mark.gpu

SHAPES = [  # layout, algorithm, n, batch
    (0, -1, 8, 300), (0, -1, 16, 64), (2, -1, 15, 300),      # one system per lane
    (0, -1, 37, 101),                                        # several short systems per wave
    (0, -1, 1024, 9), (0, -1, 1001, 9), (0, 5, 777, 5),      # tiles
    (2, -1, 64, 64), (2, -1, 60, 77), (2, 5, 300, 33), (2, 5, 1030, 9),
    (2, -1, 3001, 37), (2, -1, 2048, 64),                    # cooperative blocks
    (0, -1, 20001, 3), (0, -1, 300001, 1),
    (0, 5, 20000, 3),                                        # chunks through global memory
    (2, -1, 17000, 3),                                       # through a contiguous copy
    (0, 1, 1000, 9), (2, 1, 100, 33),                        # Thomas
]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("start", [0, 1])
def test_same_bits(prec, start):
    import torch
    import tridiagonalsolver_amd as T
    L = T.lib()
    dt = torch.float64 if prec else torch.float32
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    fails = []
    for layout, algo, n, batch in SHAPES:
        announce("solve to", prec, layout, algo, n, batch, start)
        m = n * batch
        full = [torch.rand(m + 8, device="cuda", dtype=dt) * 2 - 1 for _ in range(4)]
        full[1] = full[0].abs() + full[2].abs() + 1.5
        a, b, c, d = (t[start:start + m] for t in full)
        ref, cr = full[3].clone(), full[2].clone()
        T.check(L.tridiag_solve(prec, algo, layout, n, batch, a.data_ptr(), b.data_ptr(),
                                cr[start:].data_ptr(), ref[start:].data_ptr(), stream))
        keep = [t.clone() for t in full]
        out = torch.full_like(full[3], 7.0)
        T.check(L.tridiag_solve_to(prec, algo, layout, n, batch, a.data_ptr(), b.data_ptr(),
                                   c.data_ptr(), d.data_ptr(), out[start:].data_ptr(), None, 0,
                                   stream))
        same = torch.equal(out[start:start + m], ref[start:start + m])
        around = bool((out[:start] == 7).all() and (out[start + m:] == 7).all())
        inputs = all(torch.equal(t, k) for i, (t, k) in enumerate(zip(full, keep))
                     if algo != 1 or i != 2)
        if not (same and around and inputs):
            fails.append((layout, algo, n, batch, same, around, inputs))
    assert not fails, fails


def test_refused():
    import torch
    import tridiagonalsolver_amd as T
    from tridiagonalsolver_amd import _capi
    t = torch.zeros(4096, device="cuda")
    p, x = t.data_ptr(), torch.zeros(4096, device="cuda").data_ptr()
    L = T.lib()
    assert L.tridiag_solve_to(0, -1, 1, 64, 4, p, p, p, p, x, None, 0, None) == _capi.EUNSUPPORTED
    assert L.tridiag_solve_to(0, 0, 0, 64, 4, p, p, p, p, x, None, 0, None) == _capi.EUNSUPPORTED
    assert L.tridiag_solve_to(0, -1, 0, 64, 4, p, p, p, p, None, None, 0, None) == _capi.EINVAL


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [256, 384, 512, 768, 1024, 1536, 2048, 3072, 4096, 8192])
def test_exact_tiles(prec, n):
    """Capacities of the contiguous tiles, whose exact kernels solve in place only."""
    import torch
    import tridiagonalsolver_amd as T
    dt = torch.float64 if prec else torch.float32
    announce("solve to, exact tiles", prec, n)
    a, c, d = (torch.rand(33, n, device="cuda", dtype=dt) * 2 - 1 for _ in range(3))
    b = a.abs() + c.abs() + 1
    ref = T.solve(a, b, c, d.clone())
    keep = d.clone()
    x = T.tridiagonal_solve(a, b, c, d)
    assert torch.equal(x, ref) and torch.equal(d, keep)
