"""Solves on several threads and streams at once: their persistent kernels (panel QR, bulge chase) have
to find room beside each other."""
import threading

import pytest

import cuev_amd as cv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,threads,reps", [(1000, 6, 4), (4096, 4, 3), (8192, 4, 2)])
def test_concurrent_solves(torch_dev, n, threads, reps):
    torch = torch_dev
    mats, refs = [], []
    for t in range(threads):
        g = torch.Generator(device="cuda")
        g.manual_seed(n + t)
        G = torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64)
        mats.append((G + G.T) / 2)
        refs.append(cv.symm_eig_solve(mats[t])[0])
    torch.cuda.synchronize()
    errors = []

    def work(t):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(reps):
                    w, _ = cv.symm_eig_solve(mats[t])
                    # two runs of one solve differ by roundings at most
                    assert float((w - refs[t]).abs().max()) <= 1e-12 * float(refs[t].abs().max())
                torch.cuda.current_stream().synchronize()
        except Exception as ex:  # noqa: BLE001 (reported below, from the main thread)
            errors.append(repr(ex))

    pool = [threading.Thread(target=work, args=(t,)) for t in range(threads)]
    for x in pool:
        x.start()
    for x in pool:
        x.join()
    assert not errors
