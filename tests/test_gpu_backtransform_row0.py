"""The bulge back-transform leaves row 0, which no reflector covers, alone: what it holds has no
influence on the other rows, not even NaN or infinity."""
import numpy as np
import pytest

import cuev_amd as cv
from helpers import to_dev, from_dev, raw_put

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,b", [(3, 16), (40, 16), (130, 32), (258, 64)])
@pytest.mark.parametrize("prec", ["d", "s"])
def test_row_zero_stays_out(torch_dev, n, b, prec):
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    rng = np.random.default_rng(n)
    M0 = rng.standard_normal((n, n))
    with cv.Handle(dt, n, b, b) as h:
        Uptr, ldu = h.buffer("U")
        U = np.zeros((ldu, n))
        for s in range(n - 2):
            for r0 in range(s + 1, n, b):
                w = rng.standard_normal(min(b, n - r0))
                U[r0 - s - 1:r0 - s - 1 + len(w), s] = w / np.linalg.norm(w) if len(w) > 1 else 0.0
        raw_put(Uptr, U, dt)
        for apply in (h.bc_back, h.bc_back_t):
            out = []
            for bad in (0.0, np.nan, np.inf):
                M1 = M0.copy()
                M1[0] = bad
                M = to_dev(M1, dt)
                apply(M, n)
                torch.cuda.synchronize()
                out.append(from_dev(M))
                assert np.array_equal(out[-1][0], M1[0], equal_nan=True)
            assert np.array_equal(out[0][1:], out[1][1:]) and np.array_equal(out[0][1:], out[2][1:])
