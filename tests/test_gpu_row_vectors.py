"""Tiles that read and write 16-byte row vectors per lane, on full grids.

A 16-byte buffer store still reads its data registers while the next instruction issues;
overwritten there, single elements of a few chunks of a large launch come out wrong, which
small batches rarely show.  Every such tile solves 2^21 unknowns three times; every element
is compared with the FP64 cyclic reduction of the same systems.  Bound: the solve is
diagonally dominant (margin >= 1), so |error| <= 64 eps max|x|.
"""
import ctypes

import numpy as np
import pytest

from gpu_util import announce

pytestmark = pytest.mark.gpu


def _reference(a, b, c, d):
    """Cyclic reduction of (batch, n) systems in FP64."""
    import torch
    pad = torch.nn.functional.pad
    a, b, c, d = (t.double() for t in (a, b, c, d))
    a, c = a.clone(), c.clone()
    a[:, 0] = 0
    c[:, -1] = 0
    s, n = 1, a.shape[1]
    while s < n:
        def lo(t, v):
            return pad(t[:, :-s], (s, 0), value=v)

        def hi(t, v):
            return pad(t[:, s:], (0, s), value=v)
        k1, k2 = a / lo(b, 1.0), c / hi(b, 1.0)
        d = d - k1 * lo(d, 0.0) - k2 * hi(d, 0.0)
        b = b - k1 * lo(c, 0.0) - k2 * hi(a, 0.0)
        a, c = -k1 * lo(a, 0.0), -k2 * hi(c, 0.0)
        s *= 2
    return d / b


@pytest.mark.parametrize("prec", [0, 1])
def test_full_grids(prec):
    import torch
    import tridiagonalsolver_amd as T
    dt = torch.float64 if prec else torch.float32
    eps = np.finfo(np.float64 if prec else np.float32).eps
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    cases, fails = {}, []
    tiles = [t for t in T.tiles(prec) if t["vec"] and not t["transposed"] and not t["wide_addr"]]
    assert tiles
    for t in sorted(tiles, key=lambda t: t["cap"]):
        n = t["cap"] - (16 if t["padded"] else 0)
        announce("row vectors", prec, t["index"], n)
        if n not in cases:
            cases.clear()
            gen = torch.Generator(device="cuda").manual_seed(n)
            batch = (1 << 21) // n
            a, c, d = (torch.rand(batch, n, generator=gen, device="cuda", dtype=dt) * 2 - 1
                       for _ in range(3))
            b = a.abs() + c.abs() + 1 + torch.rand(batch, n, generator=gen, device="cuda", dtype=dt)
            cases[n] = (a, b, c, d), _reference(a, b, c, d)
        v, ref = cases[n]
        for _ in range(3):
            x = v[3].clone()
            ptrs = [ctypes.c_void_p(u.data_ptr()) for u in (v[0], v[1], v[2], x)]
            T.check(T.lib().tridiag_solve_tile(prec, t["index"], 0, n, x.shape[0], *ptrs, stream))
            err = float((x.double() - ref).abs().max() / ref.abs().max())
            if not err <= 64 * eps:
                fails.append((t["index"], t["M"], t["NW"], t["S"], n, err))
    assert not fails, fails
