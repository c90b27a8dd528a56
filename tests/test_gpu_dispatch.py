"""Solves with every option left to the library, on both sides of each line where it
changes its bandwidth, back-transform order or tridiagonal solver, against LAPACK."""
import numpy as np
import pytest
import scipy.linalg as sl

import cuev_amd as cv
from helpers import eig_metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 127, 128, 129, 130, 159, 160, 161, 255, 256, 257, 700])
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


def _small_matrix(kind, n, rng):
    """Symmetric matrices that take each way through the small solver."""
    G = rng.standard_normal((n, n))
    if kind == "random":  # one unsplit block, gaps of about 1 / n
        return (G + G.T) / 2
    if kind == "lowrank":  # T splits after rank steps: exact multiple eigenvalue
        return G[:, : max(1, n // 4)] @ G[:, : max(1, n // 4)].T + np.eye(n)
    if kind == "close":  # gaps of 1e-9: two orthogonalization steps
        Q, _ = np.linalg.qr(G)
        A = (Q * (1.0 + 1e-9 * np.arange(n))) @ Q.T
        return (A + A.T) / 2
    if kind == "pairs":  # Wilkinson's matrix: pairs closer than rounding in one block, QL
        return np.diag(np.abs(np.arange(n) - (n - 1) / 2.0)) + np.eye(n, k=1) + np.eye(n, k=-1)
    if kind == "scaled":
        return (G + G.T) * 1e170
    return np.diag(G[0])  # "diagonal"


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("kind", ["random", "lowrank", "close", "pairs", "scaled", "diagonal"])
@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 96, 113, 127, 128, 129])
def test_small_orders(torch_dev, n, kind, prec):
    """Batched, single and eigenvalues-only calls around the small solver's block and thread
    counts: LAPACK's eigenvalues, small residual and loss of orthogonality."""
    torch = torch_dev
    if kind == "scaled" and (prec == "s" or n > 128):
        pytest.skip("1e170 is not a float, and the staged pipeline squares entries without scaling")
    rng = np.random.default_rng(n)
    dt = torch.float64 if prec == "d" else torch.float32
    A = torch.from_numpy(np.stack([_small_matrix(kind, n, rng) for _ in range(3)])).to(dt)
    A64 = A.double().numpy()
    lb, Vb = cv.symm_eig_batched(A.cuda())
    # u times the sqrt(n) growth of n orthogonal transformations, with a factor for their
    # constants; FP32 results are FP64 ones rounded once
    u = 2.2e-16 if prec == "d" else 1.2e-7
    for b in range(3):
        ls, Vs = cv.symm_eig_solve(A[b].cuda())
        lv = cv.symm_eig_values(A[b].cuda())
        ref = sl.eigh(A64[b], eigvals_only=True, driver="evd")
        scale = np.abs(ref).max() or 1.0  # a zero matrix is left as it is
        for lam, V in ((lb[b], Vb[b]), (ls, Vs)):
            ev_err, res, orth = eig_metrics(A64[b] / scale, lam.double().cpu().numpy() / scale,
                                            V.double().cpu().numpy(), ref / scale)
            assert ev_err < 20 * np.sqrt(n) * u and res * n < 20 * np.sqrt(n) * u and orth < 20 * u
        assert np.abs(lv.double().cpu().numpy() - ref).max() < 20 * np.sqrt(n) * u * scale


def test_small_not_finite(torch_dev):
    """NaN and infinite entries are reported, by the batched call for its matrix only."""
    torch = torch_dev
    A = torch.eye(40, dtype=torch.float64).repeat(3, 1, 1)
    A[1, 7, 3] = float("nan")
    for bad in (float("nan"), float("inf")):
        A[1, 7, 3] = bad
        with pytest.raises(cv.CuevError) as e:
            cv.symm_eig_batched(A.cuda())
        assert e.value.status == 9
        with pytest.raises(cv.CuevError) as e:
            cv.symm_eig_solve(A[1].cuda())
        assert e.value.status == 7
        with pytest.raises(cv.CuevError) as e:
            cv.symm_eig_values(A[1].cuda())
        assert e.value.status == 7
    lam, _ = cv.symm_eig_solve(A[0].cuda())  # the counters are clean again
    assert torch.all(lam == 1.0)
