"""Orders that one kernel solves by default: any stage option keeps the staged pipeline."""
import pytest

import cuev_amd as cv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opts,staged", [({}, False), ({"dc_leaf": 16}, True), ({"dc_leaf": 100}, True),
                                         ({"bandwidth": 32}, True), ({"block": 64}, True),
                                         ({"bt_mode": "direct"}, True), ({"dc_mode": "device"}, True),
                                         ({"dc_mode": "device", "dc_leaf": 16}, True)])
@pytest.mark.parametrize("n", [20, 100, 128])
def test_stage_option_keeps_the_pipeline(torch_dev, n, opts, staged):
    torch = torch_dev
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    G = torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64)
    A = (G + G.T) / 2
    lam, V, t = cv.symm_eig_solve(A, timer=True, **opts)
    assert (t["bc_ms"] > 0) == staged  # the single kernel fills total_ms only
    ref = torch.linalg.eigvalsh(A.cpu()).cuda()
    # backward error of the solve: at most about n roundings of ||A||
    assert float((lam - ref).abs().max()) <= n * 2.3e-16 * float(ref.abs().max())
