"""Solves with every option left to the library, on both sides of each line where it
changes its bandwidth, back-transform order or tridiagonal solver, against LAPACK."""
import numpy as np
import pytest
import scipy.linalg as sl

import cuev_amd as cv
from helpers import eig_metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 159, 160, 161, 255, 256, 257, 700])
def test_auto_options(torch_dev, n, prec):
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    rng = np.random.default_rng(n)
    G = rng.standard_normal((n, n))
    A = torch.from_numpy((G + G.T) / 2).to(dt)
    ev, V = cv.symm_eig_solve(A.cuda())
    A64 = A.double().numpy()
    ref = sl.eigh(A64, eigvals_only=True, driver="evd")
    ev_err, res, orth = eig_metrics(A64, ev.double().cpu().numpy(), V.double().cpu().numpy(), ref)
    # backward error and loss of orthogonality of a two-stage solve: at most about n roundings
    u = 1.2e-16 if prec == "d" else 6e-8
    assert ev_err < 50 * np.sqrt(n) * u
    assert res < 50 * u and orth < 50 * u


@pytest.mark.parametrize("kind,n", [(k, n) for k in ("random", "split", "constant", "graded")
                                    for n in (7, 8, 9, 1024, 1025)] +
                         [("random", 2049), ("constant", 4080), ("graded", 4079), ("split", 4081), ("random", 8161)])
def test_tridi_values_stage_edges(torch_dev, kind, n):
    """Row counts around the LDS stage and the lines where the lanes per eigenvalue change;
    zero off-diagonals, equal diagonals (every pivot zero at the eigenvalue) and a graded
    matrix far from 1 in scale."""
    torch = torch_dev
    rng = np.random.default_rng(n)
    d, e = rng.standard_normal(n), rng.standard_normal(n - 1)
    if kind == "split":
        e[:: 3] = 0.0
    elif kind == "constant":
        d[:], e[:] = 2.5, 0.0
    elif kind == "graded":
        g = np.exp2(-60.0 * np.arange(n) / n) * 1e150
        d, e = d * g, e * np.sqrt(g[1:] * g[:-1]) * 0.1
    w = cv.tridi_values(torch.from_numpy(d).cuda(), torch.from_numpy(e).cuda()).cpu().numpy()
    ref = sl.eigvalsh_tridiagonal(d, e, lapack_driver="stebz")
    # both within a few ulps of ||T|| of the exact values (the stopping width), plus the
    # rounding of n rows' pivots, which enters like a change of T's entries by 4 ulps
    assert np.abs(w - ref).max() <= 20 * 2.2e-16 * (np.abs(d).max() + 2 * np.abs(e).max())
    m = n // 3
    part = cv.tridi_values(torch.from_numpy(d).cuda(), torch.from_numpy(e).cuda(), m, min(n - 1, m + 5))
    assert np.array_equal(part.cpu().numpy(), w[m: m + 6])
