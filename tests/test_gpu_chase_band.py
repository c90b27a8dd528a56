"""The stage call of the bulge chase overwrites the packed band with the tridiagonal matrix."""
import numpy as np
import pytest

import cuev_amd as cv
from helpers import raw_dev, raw_put

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("n,b", [(1, 16), (2, 16), (3, 16), (16, 16), (33, 16), (32, 32), (100, 32), (65, 64), (300, 64)])
def test_stage_chase_leaves_tridiagonal_band(torch_dev, n, b, prec):
    """Row 0 of B is d, row 1 is e, everything else is zero, exactly."""
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    rng = np.random.default_rng(n + b)
    Bp = np.zeros((2 * b, n))
    for r in range(min(b, n - 1) + 1):
        Bp[r, : n - r] = rng.standard_normal(n - r)
    with cv.Handle(dt, n, b, b) as h:
        ptr = h.buffer("B")[0]
        raw_put(ptr, Bp, dt)
        h.bc_chase()
        torch.cuda.synchronize()
        d = raw_dev(h.buffer("D")[0], n, dt)
        e = raw_dev(h.buffer("E")[0], n, dt)
        B = raw_dev(ptr, 2 * b * n, dt).reshape((2 * b, n), order="F")
    ref = np.zeros((2 * b, n))
    ref[0], ref[1, : n - 1] = d, e[: n - 1]
    assert np.array_equal(B, ref)
