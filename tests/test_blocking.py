"""Automatic bandwidth beside a block size of the caller's: what blocking a workspace is made with."""
import ctypes

import pytest

import cuev_amd as cv

INVALID_ARGUMENT = 1


def _create(n, b, k):
    """Status of a handle's creation. Without a GPU it ends at the first HIP call, after the blocking."""
    h = ctypes.c_void_p(0)
    st = cv.lib().cuev_handle_create(ctypes.byref(h), 1, n, b, k, None)
    if h:
        p, ld = ctypes.c_void_p(0), ctypes.c_int64(0)
        assert cv.lib().cuev_handle_buffer(h, cv.BUF["B"], ctypes.byref(p), ctypes.byref(ld)) == 0
        cv.lib().cuev_handle_destroy(h)
        return st, ld.value // 2
    return st, None


@pytest.mark.parametrize("n", [255, 256, 1000, 4095])
@pytest.mark.parametrize("k", [32, 96, 160, 480])
def test_block_of_32s_is_accepted_below_4096(n, k):
    st, b = _create(n, 0, k)
    assert st != INVALID_ARGUMENT
    assert b in (None, 32)


@pytest.mark.parametrize("n,k", [(255, 48), (256, 16), (1000, 33), (4096, 32), (4096, 96), (5000, 480)])
def test_other_blocks_stay_refused(n, k):
    assert _create(n, 0, k)[0] == INVALID_ARGUMENT


@pytest.mark.gpu
@pytest.mark.parametrize("n,k,b", [(255, 0, 32), (255, 64, 32), (256, 0, 64), (256, 64, 64), (300, 96, 32), (1000, 128, 64),
                                   (4095, 96, 32), (4096, 64, 64)])
def test_automatic_bandwidth(torch_dev, n, k, b):
    assert _create(n, 0, k) == (0, b)


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(300, 32), (300, 96)])
def test_solve_with_block_of_32s(torch_dev, n, k):
    torch = torch_dev
    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    G = torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64)
    A = (G + G.T) / 2
    lam, V = cv.symm_eig_solve(A, block=k)
    ref = torch.linalg.eigvalsh(A.cpu()).cuda()
    # backward error of a two-stage solve: at most about n roundings of ||A||
    tol = n * 2.3e-16 * float(ref.abs().max())
    assert float((lam - ref).abs().max()) <= tol
    assert float((A @ V - V * lam).norm(dim=0).max()) <= tol * n ** 0.5
    assert float((cv.symm_eig_values(A, block=k) - ref).abs().max()) <= tol
