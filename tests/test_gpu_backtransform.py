"""The bulge back-transform at the edges of its passes (4 or 8 hops, a wave each), its sweep groups
and its column strips, against the oracle's reflector-by-reflector order."""
import numpy as np
import pytest

import cuev_amd as cv
from helpers import to_dev, from_dev, raw_put
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,b", [(3, 16), (17, 16), (18, 16), (19, 16), (65, 16), (66, 16), (129, 16), (130, 16),
                                 (131, 32), (257, 32), (258, 32), (291, 32), (67, 64), (257, 64), (258, 64),
                                 (513, 64), (514, 64), (611, 64)])
@pytest.mark.parametrize("prec", ["d", "s"])
def test_bc_back_edges(torch_dev, n, b, prec):
    """Random reflectors in every hop. Tolerance: a row meets about n of them; 64 units of rounding
    each bounds the entries of the orthogonal result."""
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    rng = np.random.default_rng(n + b)
    with cv.Handle(dt, n, b, b) as h:
        Uptr, ldu = h.buffer("U")
        U = np.zeros((ldu, n))
        for s in range(n - 2):
            for r0 in range(s + 1, n, b):
                w = rng.standard_normal(min(b, n - r0))
                U[r0 - s - 1:r0 - s - 1 + len(w), s] = w / np.linalg.norm(w) if len(w) > 1 else 0.0
        raw_put(Uptr, U, dt)
        Q, QT = to_dev(np.eye(n), dt), to_dev(np.eye(n), dt)
        h.bc_back(Q, n)
        h.bc_back_t(QT, n)
        torch.cuda.synchronize()
        Q, QT = from_dev(Q), from_dev(QT)
    U = U.astype(np.float64 if prec == "d" else np.float32).astype(np.float64)
    ref = O.bc_back(np.asfortranarray(U), np.eye(n, order="F"), b)
    tol = 64 * n * (2.0 ** -53 if prec == "d" else 2.0 ** -24)
    assert np.abs(Q - ref).max() <= tol
    assert np.abs(QT - ref.T).max() <= tol
