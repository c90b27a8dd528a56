"""Products whose last tile columns are split off and divided along K: a few tiles more than whole
rounds over the CUs, with odd edges, both operand orders of each kind and beta."""
import pytest

import cuev_amd as cv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(3000, 3000, 1024), (2945, 3001, 1031), (4096, 2177, 1500), (2817, 3080, 2048),
                                   (3000, 2690, 1023), (6000, 2200, 1100)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("prec", ["d", "s"])
def test_gemm_tail_columns(torch_dev, M, N, K, ta, tb, prec):
    torch = torch_dev
    dt = torch.float64 if prec == "d" else torch.float32
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K)
    A = torch.randn((K, M) if not ta else (M, K), generator=g, device="cuda", dtype=dt)  # op(A)'s columns as rows
    B = torch.randn((N, K) if not tb else (K, N), generator=g, device="cuda", dtype=dt)
    C0 = torch.randn((N, M), generator=g, device="cuda", dtype=dt)
    C = C0.clone()
    cv.gemm(ta, tb, M, N, K, 0.5, A, M if not ta else K, B, K if not tb else N, -2.0, C, M)
    a, b = (A if not ta else A.T).double(), (B if not tb else B.T).double()  # K x M, N x K
    ref = 0.5 * (b @ a) - 2.0 * C0.double()
    u = 2.0 ** -53 if prec == "d" else 2.0 ** -24
    bound = (K + 8) * u * (0.5 * (b.abs() @ a.abs()) + 2.0 * C0.double().abs())
    assert bool(((C.double() - ref).abs() <= bound).all())
