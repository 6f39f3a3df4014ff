"""Interleaved tiles that read whole 128-byte row pieces, at any number of rows and systems.

Sizes on both sides of every capacity, batches that leave the last group of systems partial
and rows that start on and off 128-byte lines, in arrays that start at any element with NaN
around them.  Bound: the systems are diagonally dominant with margin >= 1, so
|error| <= 64 eps max|x| against FP64 cyclic reduction of the same systems.
"""
import numpy as np
import pytest

from gpu_util import announce

pytestmark = pytest.mark.gpu

PAD = 37


def _reference(a, b, c, d):
    """Cyclic reduction of interleaved (n, batch) systems in FP64."""
    import torch
    a, b, c, d = (t.double().clone() for t in (a, b, c, d))
    a[0] = 0
    c[-1] = 0
    s, n = 1, a.shape[0]
    while s < n:
        def lo(t, v):
            return torch.cat([t.new_full((s, t.shape[1]), v), t[:-s]])

        def hi(t, v):
            return torch.cat([t[s:], t.new_full((s, t.shape[1]), v)])
        k1, k2 = a / lo(b, 1.0), c / hi(b, 1.0)
        d = d - k1 * lo(d, 0.0) - k2 * hi(d, 0.0)
        b = b - k1 * lo(c, 0.0) - k2 * hi(a, 0.0)
        a, c = -k1 * lo(a, 0.0), -k2 * hi(c, 0.0)
        s *= 2
    return d / b


def _embedded(t, start):
    """t inside a buffer of NaN, from element `start`."""
    import torch
    buf = torch.full((start + t.numel() + PAD,), float("nan"), device="cuda", dtype=t.dtype)
    view = buf[start:start + t.numel()].view_as(t)
    view.copy_(t)
    return buf, view


def check_interleaved(dt, n, batch, start, plan_kind=None):
    """Relative error of one solve (inf when memory around d changed)."""
    import torch
    import tridiagonalsolver_amd as T
    from tridiagonalsolver_amd import _capi
    if plan_kind is not None:
        assert _capi.plan(0 if dt == torch.float32 else 1, -1, 2, n, batch)["kind"] == plan_kind
    gen = torch.Generator(device="cuda").manual_seed(n * 1000 + batch)
    a, c, d = (torch.rand(n, batch, generator=gen, device="cuda", dtype=dt) * 2 - 1
               for _ in range(3))
    b = a.abs() + c.abs() + 1 + torch.rand(n, batch, generator=gen, device="cuda", dtype=dt)
    ref = _reference(a, b, c, d)
    bufs, views = zip(*(_embedded(t, start) for t in (a, b, c, d)))
    T.solve(*views, layout=T.INTERLEAVED)
    around = torch.cat([bufs[3][:start], bufs[3][start + n * batch:]])
    if not bool(around.isnan().all()):
        return float("inf")
    err = float((views[3].double() - ref).abs().max() / ref.abs().max())
    return err if err == err else float("inf")


@pytest.mark.parametrize("prec", [0, 1])
def test_any_size(prec):
    import torch
    dt = torch.float64 if prec else torch.float32
    S = 16 if prec else 32
    caps = (32, 48, 64, 96, 128, 192, 256, 384, 512)
    sizes = sorted({n for cap in caps for n in (cap - 1, cap, cap + 1) if 17 <= n <= 512})
    fails = []
    for n in sizes:
        for batch, start in ((1, 0), (S - 1, 1), (4 * S, 0), (4 * S, 3), (17 * S + 5, 1)):
            announce("interleaved pieces", prec, n, batch, start)
            err = check_interleaved(dt, n, batch, start)
            if not err <= 64 * np.finfo(np.float64 if prec else np.float32).eps:
                fails.append((n, batch, start, err))
    assert not fails, fails


@pytest.mark.parametrize("prec", [0, 1])
def test_full_grids(prec):
    """Enough systems that several tiles share every XCD, rows on and off lines."""
    import torch
    dt = torch.float64 if prec else torch.float32
    eps = np.finfo(np.float64 if prec else np.float32).eps
    errs = {(n, batch): check_interleaved(dt, n, batch, 0)
            for n, batch in ((60, 20000), (60, 20001), (100, 12345), (200, 8191), (400, 4100))}
    assert all(e <= 64 * eps for e in errs.values()), errs
