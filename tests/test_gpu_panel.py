"""Panel QR where its kernel's shapes change: two or three sets of lanes for the rows under the
Gram matrix, slices of 64, 80 and 96 rows with partial last slices, one or several workgroups,
and a second Cholesky pass that is, or is not, close to the identity."""
import numpy as np
import pytest

import cuev_amd as cv
from helpers import to_dev, from_dev, raw_dev, empty_dev
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,b", [(65, 64), (100, 64), (33, 32), (17, 16), (128, 64), (129, 64), (191, 64), (16385, 64), (20487, 64), (64, 32), (97, 32),
                                    (16401, 32), (32, 16), (65, 16), (20481, 16)])
@pytest.mark.parametrize("cond", [1.0, 1e4])
@pytest.mark.parametrize("prec", ["d", "s"])
def test_panel_qr_edges(torch_dev, rows, b, cond, prec):
    """A = Q R with Q = I - Y T Y^T orthogonal, and the reflectors in LAPACK's form (unit lower
    trapezoidal, tau in [1, 2]). Tolerance: 64 units of rounding per column, for the products of b
    reflectors (the Gram route adds none: two passes)."""
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    rng = np.random.default_rng(rows + b)
    A0 = rng.standard_normal((rows, b)) @ np.diag(np.logspace(0, -np.log10(cond), b)) @ np.linalg.qr(
        rng.standard_normal((b, b)))[0]
    A0 = A0.astype(np.float64 if prec == "d" else np.float32).astype(np.float64)
    with cv.Handle(dt, rows, b, b) as h:
        dA, dY = to_dev(A0, dt), empty_dev(rows, b, dt)
        h.dbbr_panel_qr(dA, dY, rows, b)
        torch.cuda.synchronize()
        Af, Y = from_dev(dA).astype(np.float64), from_dev(dY).astype(np.float64)
        T = raw_dev(h.buffer("TRI")[0], b * b, dt).reshape((b, b), order="F").astype(np.float64)
        tau = raw_dev(h.buffer("TAU")[0], b, dt).astype(np.float64)
    tol = 64 * b * (2.0 ** -53 if prec == "d" else 2.0 ** -24)
    R = np.zeros_like(A0)
    R[:b] = np.triu(Af[:b])
    assert np.linalg.norm(R - Y @ (T @ (Y.T @ R)) - A0) <= tol * np.linalg.norm(A0)
    Qb = np.eye(rows, b) - Y @ (T @ Y[:b].T)
    assert np.linalg.norm(Qb.T @ Qb - np.eye(b)) <= tol * np.sqrt(b)
    assert np.array_equal(np.tril(Y[:b], -1), np.tril(Af[:b], -1)) and np.array_equal(Y[b:], Af[b:])
    assert np.all(np.diag(Y[:b]) == 1) and np.all(np.triu(Y[:b], 1) == 0) and np.all(np.tril(T, -1) == 0)
    assert np.array_equal(tau, np.diag(T)) and np.all(tau >= 1 - tol) and np.all(tau <= 2 + tol)


@pytest.mark.parametrize("rows,b", [(1, 64), (2, 64), (63, 64), (64, 64), (1, 32), (32, 32), (15, 16), (16, 16)])
def test_panel_qr_last_panels(torch_dev, rows, b):
    """Panels of at most b rows: the Householder kernel in one workgroup, ending at the last row."""
    torch = torch_dev
    A0 = np.random.default_rng(rows + b).standard_normal((rows, b))
    with cv.Handle(torch.float64, rows, b, b) as h: # its order is the panel's leading dimension
        dA, dY = to_dev(A0, torch.float64), empty_dev(rows, b, torch.float64)
        h.dbbr_panel_qr(dA, dY, rows, b)
        torch.cuda.synchronize()
        Af, Y = from_dev(dA), from_dev(dY)
        T = raw_dev(h.buffer("TRI")[0], b * b, torch.float64).reshape((b, b), order="F")
        tau = raw_dev(h.buffer("TAU")[0], b, torch.float64)
    Ao, Yo, To, tauo = O.panel_qr(A0, b)
    tol = 64 * b * 2.0 ** -53
    m = min(rows, b)
    assert np.abs(np.triu(Af) - np.triu(Ao)).max() <= tol * np.abs(A0).max() * np.sqrt(rows)
    assert np.abs(Y - Yo).max() <= tol and np.abs(T[:m, :m] - To[:m, :m]).max() <= 2 * tol
    assert np.abs(tau - tauo).max() <= tol
    assert np.all(T[:, m:] == 0) and np.all(T[m:] == 0) and np.all(tau[m:] == 0)
