"""The windowed bulge chase, which orders take whose resident form does not fit on the GPU: the same
edges as the resident one, several phases of its schedule, and both forms on one handle."""
import numpy as np
import pytest

import cuev_amd as cv
from helpers import raw_dev, raw_put
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _band(n, b, prec, seed):
    rng = np.random.default_rng(seed)
    Bp = np.zeros((2 * b, n))
    for r in range(min(b, n - 1) + 1):
        Bp[r, : n - r] = rng.standard_normal(n - r)
    return Bp.astype(np.float64 if prec == "d" else np.float32).astype(np.float64)


def _chase(torch, h, Bp, dt):
    n, b = h.n, h.nbw
    ptr = h.buffer("B")[0]
    raw_put(ptr, Bp, dt)
    h.bc_chase()
    torch.cuda.synchronize()
    Uptr, ldu = h.buffer("U")
    return (raw_dev(h.buffer("D")[0], n, dt), raw_dev(h.buffer("E")[0], n, dt),
            raw_dev(Uptr, ldu * n, dt).reshape((ldu, n), order="F"),
            raw_dev(ptr, 2 * b * n, dt).reshape((2 * b, n), order="F"))


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("b", [16, 32, 64])
@pytest.mark.parametrize("blocks,extra", [(0, 3), (0, 5), (1, 0), (1, 1), (1, 2), (1, 3), (2, 1), (2, 2), (4, 0),
                                          (4, 1), (5, 3)])
def test_windowed_chase_edges(torch_dev, b, blocks, extra, prec):
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    n = blocks * b + extra
    Bp = _band(n, b, prec, 100 * b + n)
    ref = O.bc_chase(np.asfortranarray(Bp), b)
    # the stage tests' tolerances: an intermediate reflector may amplify a rounding by the inverse
    # of a small tail
    tol = 1e-9 if prec == "d" else 2e-2
    scale = max(1.0, np.abs(ref["d"]).max())
    with cv.Handle(dt, n, b, max(b, 64)) as h:
        h.set_chase(windowed=True)
        for _ in range(2):
            d, e, U, B = _chase(torch, h, Bp, dt)
            assert np.abs(d - ref["d"]).max() / scale < tol
            assert np.abs(np.abs(e[: n - 1]) - np.abs(ref["e"][: n - 1])).max() / scale < tol
            assert e[n - 1] == 0.0
            for sw in range(n - 2):
                assert np.abs(U[: n - 1 - sw, sw] - ref["U"][: n - 1 - sw, sw]).max() < 10 * tol
                assert np.all(U[n - 1 - sw: n, sw] == 0.0)
            assert np.array_equal(B[0], d) and np.array_equal(B[1, : n - 1], e[: n - 1])
            assert B[1, n - 1] == 0.0 and np.all(B[2:] == 0.0)


@pytest.mark.parametrize("n,b", [(600, 16), (1500, 32), (2500, 64)])
@pytest.mark.parametrize("prec", ["d", "s"])
def test_both_forms_agree(torch_dev, n, b, prec):
    """Several hundred sweeps (up to eight phases): the eigenvalues of the two tridiagonal matrices
    agree within the n roundings of ||B|| each of them may be off by."""
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    Bp = _band(n, b, prec, n)
    lam = []
    with cv.Handle(dt, n, b, b) as h:
        for windowed in (False, True, False):
            h.set_chase(windowed=windowed)
            d, e = _chase(torch, h, Bp, dt)[:2]
            lam.append(cv.tridi_values(torch.from_numpy(d).cuda(), torch.from_numpy(e).cuda()).cpu().numpy())
    u = 2.0 ** -53 if prec == "d" else 2.0 ** -24
    tol = 2 * n * u * np.abs(lam[0]).max()
    assert np.abs(lam[0] - lam[1]).max() <= tol and np.array_equal(lam[0], lam[2])


@pytest.mark.parametrize("n,b", [(9000, 16), (17000, 32), (17000, 64)])
@pytest.mark.parametrize("prec", ["d", "s"])
def test_resident_without_receiving_wave(torch_dev, n, b, prec):
    """Orders above half of what the GPU holds of the chase with a receiving wave (256 CUs: n = 8192 at
    b = 16, 16384 at b = 32 and 64 in FP64) take the form without it: eigenvalues against the windowed form."""
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    Bp = _band(n, b, prec, n)
    lam = []
    with cv.Handle(dt, n, b, b) as h:
        for windowed in (False, True):
            h.set_chase(windowed=windowed)
            raw_put(h.buffer("B")[0], Bp, dt)
            h.bc_chase()
            torch.cuda.synchronize()
            d, e = (raw_dev(h.buffer(x)[0], n, dt) for x in "DE")
            lam.append(cv.tridi_values(torch.from_numpy(d).cuda(), torch.from_numpy(e).cuda()).cpu().numpy())
    u = 2.0 ** -53 if prec == "d" else 2.0 ** -24
    # each within n roundings of ||B||
    assert np.abs(lam[0] - lam[1]).max() <= 2 * n * u * np.abs(lam[0]).max()


def test_form_is_checked(torch_dev):
    """A null handle and another value than 0 or 1 are refused."""
    assert cv.lib().cuev_handle_set_chase(None, 1) == 1
    with cv.Handle(torch_dev.float32, 10, 16, 16) as h:
        assert cv.lib().cuev_handle_set_chase(h.h, 2) == 1
