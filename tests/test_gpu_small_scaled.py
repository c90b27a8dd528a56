"""Matrices of order <= 128 whose eigenvalues agree to many digits, at every scale of their type: a
single solve is as good as a batched one, whichever way it takes."""
import numpy as np
import pytest
import scipy.linalg as sl

import cuev_amd as cv
from helpers import eig_metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,exp", [("d", x) for x in (-900, -565, -301, -300, 0, 299, 300, 301, 565, 1000)] +
                         [("s", x) for x in (-110, -101, -100, 0, 99, 100, 101, 115)])
@pytest.mark.parametrize("dense", [True, False])
@pytest.mark.parametrize("n", [33, 48, 64, 65, 128])
def test_close_pairs_at_any_scale(torch_dev, n, dense, prec, exp):
    """Wilkinson's matrix, as it is or under one reflection that leaves its first row (the reduction
    finds a tridiagonal form that does not split), times 2^exp. Its eigenvalues are the unscaled ones
    times 2^exp, and each call's errors those of an unscaled solve (20 sqrt(n) roundings of ||A||, as
    for all small orders)."""
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    A1 = np.diag(np.abs(np.arange(n) - (n - 1) / 2.0)) + np.eye(n, k=1) + np.eye(n, k=-1)
    if dense:
        v = np.random.default_rng(n).standard_normal(n)
        v[0] = 0.0
        P = np.eye(n) - 2.0 * np.outer(v, v) / (v @ v)
        A1 = P @ A1 @ P
        A1 = (A1 + A1.T) / 2
    A1 = A1.astype(np.float64 if prec == "d" else np.float32).astype(np.float64)
    A = torch.from_numpy(np.ldexp(A1, exp)).to(dt)
    ref = sl.eigvalsh(A1)
    u = 2.2e-16 if prec == "d" else 1.2e-7
    single, batched = cv.symm_eig_solve(A.cuda()), cv.symm_eig_batched(A[None].cuda())
    for lam, V in (single, (batched[0][0], batched[1][0])):
        lam1 = np.ldexp(lam.double().cpu().numpy(), -exp)
        ev_err, res, orth = eig_metrics(A1, lam1, V.double().cpu().numpy(), ref)
        assert ev_err < 20 * np.sqrt(n) * u and res * n < 20 * np.sqrt(n) * u and orth < 20 * u
    lv = np.ldexp(cv.symm_eig_values(A.cuda()).double().cpu().numpy(), -exp)
    assert np.abs(lv - ref).max() < 20 * np.sqrt(n) * u * np.abs(ref).max()
