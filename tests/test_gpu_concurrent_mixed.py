"""Solves of different sizes at once, and stage calls beside them: their persistent kernels (panel QR,
bulge chase) all find room."""
import threading

import pytest

import cuev_amd as cv

pytestmark = pytest.mark.gpu


def _run_all(torch, jobs):
    errors = []

    def work(job):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                job()
                torch.cuda.current_stream().synchronize()
        except Exception as ex:  # noqa: BLE001 (reported below, from the main thread)
            errors.append(repr(ex))

    pool = [threading.Thread(target=work, args=(j,)) for j in jobs]
    for x in pool:
        x.start()
    for x in pool:
        x.join()
    assert not errors


def _solver(torch, n, seed, reps, values=False):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    G = torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64)
    A = (G + G.T) / 2
    ref = cv.symm_eig_solve(A)[0]

    def job():
        for _ in range(reps):
            w = cv.symm_eig_values(A) if values else cv.symm_eig_solve(A)[0]
            # both are within about n roundings of ||A|| of the exact eigenvalues
            assert float((w - ref).abs().max()) <= n * 2.3e-16 * float(ref.abs().max())

    return job


@pytest.mark.parametrize("sizes", [((8192, 2), (4096, 3), (4096, 3), (4096, 3)), ((16384, 1), (1000, 12)),
                                   ((5000, 3), (2500, 4), (300, 12), (8192, 2))])
def test_unequal_solves(torch_dev, sizes):
    torch = torch_dev
    jobs = [_solver(torch, n, n + i, reps, values=i % 2 == 1) for i, (n, reps) in enumerate(sizes)]
    torch.cuda.synchronize()
    _run_all(torch, jobs)


def test_stage_calls_beside_a_solve(torch_dev):
    torch = torch_dev
    n = 4096
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    G = torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64)
    A = (G + G.T) / 2

    def stages():
        with cv.Handle(torch.float64, n, 64, 512) as h:
            for _ in range(3):
                h.dbbr_reduce(A.clone())
                h.bc_chase()

    solve = _solver(torch, 8192, 1, 2)
    torch.cuda.synchronize()
    _run_all(torch, [solve, stages, stages])
