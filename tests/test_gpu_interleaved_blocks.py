"""Interleaved systems of more than 512 rows in cooperative row blocks, at any number of rows
and systems: blocks that end inside the last one, groups of systems that are partial, rows
on and off 128-byte lines, arrays at any element.  Bound as for the short interleaved tiles:
|error| <= 64 eps max|x| for systems of margin >= 1."""
import numpy as np
import pytest

from gpu_util import announce
from test_gpu_interleaved_pieces import check_interleaved

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [513, 767, 1023, 1025, 2100, 4097, 8191, 16384 - 255])
def test_any_size(prec, n):
    import torch
    import tridiagonalsolver_amd as T
    dt = torch.float64 if prec else torch.float32
    S = 16 if prec else 32
    fails = []
    for batch, start in ((1, 0), (S + 1, 1), (3 * S, 3), (9 * S + 5, 0)):
        announce("interleaved blocks", prec, n, batch, start)
        assert T.plan(prec, -1, 2, n, batch)["K"] == -(-n // 256)
        err = check_interleaved(dt, n, batch, start)
        if not err <= 64 * np.finfo(np.float64 if prec else np.float32).eps:
            fails.append((n, batch, start, err))
    assert not fails, fails


@pytest.mark.parametrize("prec,n,batch", [(0, 600, 20001), (0, 3001, 4096), (1, 3001, 1001),
                                          (1, 1100, 5003), (0, 9001, 777)])
def test_several_rounds(prec, n, batch):
    """More tasks than workgroups are resident, the last round partial."""
    import torch
    announce("interleaved blocks, rounds", prec, n, batch)
    err = check_interleaved(torch.float64 if prec else torch.float32, n, batch, 0)
    assert err <= 64 * np.finfo(np.float64 if prec else np.float32).eps
