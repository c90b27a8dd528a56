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
