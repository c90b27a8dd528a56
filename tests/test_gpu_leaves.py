"""The divide and conquer's leaves on the GPU, through the tridiagonal solver: leaf orders around the
largest, and tridiagonal matrices that take each way through the leaf solver (split blocks, zero
leaves, clustered eigenvalues that go to QL, leaves far from each other in scale)."""
import numpy as np
import pytest
import scipy.linalg as sl

import cuev_amd as cv
from helpers import to_dev, from_dev, empty_dev

pytestmark = pytest.mark.gpu


def _tridiagonal(kind, n, rng):
    d, e = rng.standard_normal(n), rng.standard_normal(n - 1) if n > 1 else np.zeros(0)
    if kind == "split":
        e[::3] = 0.0
    elif kind == "zero":
        d[:], e[:] = 0.0, 0.0
        d[n // 2:] = rng.standard_normal(n - n // 2)
    elif kind == "wilkinson":  # pairs of eigenvalues that agree to many digits
        d, e = np.abs(np.arange(n) % 63 - 31.0), np.ones(max(n - 1, 0))
    elif kind == "graded":
        g = np.exp2(-200.0 * np.arange(n) / n)
        d, e = d * g, e * np.sqrt(g[1:] * g[:-1]) * 0.1
    return d, e


@pytest.mark.parametrize("kind", ["random", "split", "zero", "wilkinson", "graded"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 300])
@pytest.mark.parametrize("prec", ["d", "s"])
def test_leaves(torch_dev, kind, n, prec):
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    rng = np.random.default_rng(n)
    d, e = _tridiagonal(kind, n, rng)
    if prec == "s":
        d, e = d.astype(np.float32).astype(np.float64), e.astype(np.float32).astype(np.float64)
    with cv.Handle(dt, n, 16, 16) as h:
        h.set_dc("device", 0)
        dd, de = to_dev(d, dt), to_dev(np.append(e, 0.0), dt)
        lam, Q = to_dev(np.zeros(n), dt), empty_dev(n, n, dt)
        h.tridi_dc(dd, de, lam, Q)
        torch.cuda.synchronize()
        lam, Q = from_dev(lam), from_dev(Q).reshape(n, n)
    T = np.diag(d) + (np.diag(e, 1) + np.diag(e, -1) if n > 1 else 0.0)
    u = 2.0 ** -53 if prec == "d" else 2.0 ** -24
    nrm = max(np.abs(d).max() + (2 * np.abs(e).max() if n > 1 else 0.0), 1e-300)
    # the deflation tolerance (8 u ||T||) per level of the tree, and a few roundings per row
    tol = 64 * u * np.sqrt(n)
    assert np.all(np.diff(lam) >= 0)
    assert np.abs(lam - sl.eigvalsh(T)).max() <= tol * nrm
    assert np.linalg.norm(T @ Q - Q * lam) <= tol * nrm * np.sqrt(n)
    assert np.linalg.norm(Q.T @ Q - np.eye(n)) <= tol * np.sqrt(n)
