"""The resident bulge chase at the edges of its blocks: orders of one to a few blocks plus
0 to 3 rows, every bandwidth and both precisions, against the oracle's chase of the same
band (d, |e|, every reflector)."""
import numpy as np
import pytest

import cuev_amd as cv
from helpers import raw_dev, raw_put
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("b", [16, 32, 64])
@pytest.mark.parametrize("blocks,extra", [(0, 3), (0, 5), (1, 0), (1, 1), (1, 2), (1, 3), (2, 1), (2, 2), (4, 0),
                                          (4, 1), (5, 3)])
def test_chase_edges(torch_dev, b, blocks, extra, prec):
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    n = blocks * b + extra
    rng = np.random.default_rng(100 * b + n)
    Bp = np.zeros((2 * b, n))
    for r in range(min(b, n - 1) + 1):
        Bp[r, : n - r] = rng.standard_normal(n - r)
    Bp = Bp.astype(np.float64 if prec == "d" else np.float32).astype(np.float64)
    with cv.Handle(dt, n, b, max(b, 64)) as h:
        for _ in range(2):  # again on the same buffers: no message of the first chase is taken for a new one
            raw_put(h.buffer("B")[0], Bp, dt)
            h.bc_chase()
            torch.cuda.synchronize()
            d = raw_dev(h.buffer("D")[0], n, dt)
            e = raw_dev(h.buffer("E")[0], n, dt)
            Uptr, ldu = h.buffer("U")
            U = raw_dev(Uptr, ldu * n, dt).reshape((ldu, n), order="F")
            ref = O.bc_chase(np.asfortranarray(Bp), b)
            # the chase is a sequence of about n^2 / b orthogonal transformations whose
            # intermediate reflectors may amplify a rounding by the inverse of a small
            # reflector tail: the tolerances of the stage tests
            tol = 1e-9 if prec == "d" else 2e-2
            scale = max(1.0, np.abs(ref["d"]).max())
            assert np.abs(d - ref["d"]).max() / scale < tol
            assert np.abs(np.abs(e[: n - 1]) - np.abs(ref["e"][: n - 1])).max() / scale < tol
            assert e[n - 1] == 0.0
            for sw in range(n - 2):
                assert np.abs(U[: n - 1 - sw, sw] - ref["U"][: n - 1 - sw, sw]).max() < 10 * tol
                assert np.all(U[n - 1 - sw: n, sw] == 0.0)
