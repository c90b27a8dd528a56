"""The work a user of this package has it do: inputs, one pass, and the exact results.

Families (the "op" of a case):

  solve     all eigenpairs of one FP64 matrix (``symm_eig_solve``), eigenvectors in the
            sign convention "components sum to a non-negative value"
  psd       nearest positive semidefinite matrix in FP32: eigensolve, negative eigenvalues
            cut, and V diag(max(lam, 0)) V^T as one product (``symm_eig_solve``, ``gemm``)
  grad      a training step through ``autograd.eigh`` in FP64: loss w . lam + ||V_k^T B||_F^2,
            its gradient with respect to A
  values    eigenvalues only, all or an index range (``symm_eig_values``), FP64 or FP32
  batched   all eigenpairs of many small FP64 matrices (``symm_eig_batched``)
  sqrtm     square roots of many small FP32 covariances from ``symm_eig_batched``
  backward  ``eig_backward`` on saved (lam, V) in FP32, full cotangents

Input kinds: "goe", (G + G^T) / 2 scaled to a spectrum of about [-1, 1] (the random dense
matrices of the benchmark configurations), and "cov", the covariance of 2 n samples.
"""
import math

import torch

import cuev_amd as cv
from cuev_amd import autograd

DTYPE = {"f64": torch.float64, "f32": torch.float32}


def listed():
    return [
        # one small dense problem per call, e.g. a normal-mode analysis of a molecule:
        # launches and latencies count
        {"name": "solve_48", "op": "solve", "kind": "goe", "n": 48},
        # a few hundred, odd: below the device D&C's and the reordered order's sizes
        {"name": "solve_333", "op": "solve", "kind": "cov", "n": 333},
        # the small configuration of the benchmark, with its bandwidth and block size
        {"name": "solve_1024", "op": "solve", "kind": "goe", "n": 1024, "b": 32, "k": 256},
        # an ordinary size that is no multiple of any tile
        {"name": "solve_2500", "op": "solve", "kind": "cov", "n": 2500},
        # the headline size of the benchmark
        {"name": "solve_16384", "op": "solve", "kind": "goe", "n": 16384},
        # covariance repair / an SDP's projection step in single precision
        {"name": "psd_1000_f32", "op": "psd", "kind": "goe", "n": 1000},
        # a training step at the benchmark's differentiation size: solve and backward
        {"name": "grad_4096", "op": "grad", "kind": "goe", "n": 4096, "rank": 128},
        # a whole spectrum without vectors (density of states)
        {"name": "values_8192", "op": "values", "kind": "goe", "dtype": "f64", "n": 8192, "lo": 0, "hi": 8191},
        # the largest tenth of the eigenvalues of an odd-sized covariance (how many
        # components to keep), single precision
        {"name": "values_3001_f32", "op": "values", "kind": "cov", "dtype": "f32", "n": 3001, "lo": 2700, "hi": 3000},
        # many tiny Hessians / structure tensors
        {"name": "batched_32", "op": "batched", "kind": "goe", "n": 32, "batch": 2048},
        # preconditioner blocks of a second-order optimiser, single precision
        {"name": "sqrtm_100_f32", "op": "sqrtm", "kind": "cov", "n": 100, "batch": 256},
        # the backward pass alone, single precision, a size that is no multiple of a tile
        {"name": "backward_3000_f32", "op": "backward", "n": 3000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["solve", "solve", "solve", "psd", "grad", "values", "values", "batched", "batched", "sqrtm",
                     "backward"])
    kind = rng.choice(["goe", "cov"])
    if op == "solve":
        return {"op": op, "kind": kind, "n": _log_int(rng, 16, 12000)}
    if op == "psd":
        return {"op": op, "kind": "goe", "n": _log_int(rng, 64, 4000)}
    if op == "grad":
        n = _log_int(rng, 64, 5000)
        return {"op": op, "kind": "goe", "n": n, "rank": max(1, n // 32)}
    if op == "values":
        n = _log_int(rng, 64, 10000)
        lo, hi = 0, n - 1
        if rng.random() < 0.5:  # one end of the spectrum
            m = max(1, n // rng.randint(4, 40))
            lo, hi = (0, m - 1) if rng.random() < 0.5 else (n - m, n - 1)
        return {"op": op, "kind": kind, "dtype": rng.choice(["f64", "f32"]), "n": n, "lo": lo, "hi": hi}
    if op in ("batched", "sqrtm"):
        # up to about 4 million matrix entries per call
        n = _log_int(rng, 3, 256 if op == "batched" else 160)
        return {"op": op, "kind": kind if op == "batched" else "cov", "n": n,
                "batch": max(1, min(20000, int((4 << 20) / (n * n) * rng.uniform(0.1, 1.0))))}
    return {"op": "backward", "n": _log_int(rng, 64, 6000)}


def _matrices(kind, n, batch, seed):
    """batch symmetric FP64 matrices (batch, n, n)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if kind == "goe":
        G = torch.randn((batch, n, n), generator=g, device="cuda", dtype=torch.float64)
        G.mul_(1.0 / math.sqrt(2.0 * n))  # spectrum of (G + G^T) / 2 in about [-1, 1]
        out = G + G.mT
        return out.mul_(0.5 * math.sqrt(2.0))
    X = torch.randn((batch, n, 2 * n), generator=g, device="cuda", dtype=torch.float64)
    # features of different variance, as measured data have them
    X.mul_(torch.linspace(0.5, 1.5, n, device="cuda", dtype=torch.float64)[None, :, None])
    C = torch.matmul(X, X.mT) / (2.0 * n)
    return (C + C.mT) * 0.5


def prepare(case, seed):
    op, n = case["op"], case["n"]
    if op in ("batched", "sqrtm"):
        A = _matrices(case["kind"], n, case["batch"], seed)
        return {"case": case, "A": A if op == "batched" else A.float()}
    if op == "backward":
        # a random orthogonal V, an ordered spectrum of repelling neighbours, random cotangents
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        G = torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64)
        V = torch.linalg.qr(G)[0].float()
        jitter = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * 0.5
        lam = ((torch.arange(n, device="cuda", dtype=torch.float64) + jitter) * (2.0 / n) - 1.0).float()
        Vbar = torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64).float()
        lambar = torch.randn(n, generator=g, device="cuda", dtype=torch.float64).float()
        # saved by the forward pass: V with its columns contiguous
        return {"case": case, "V": V.mT.contiguous().mT, "lam": lam, "Vbar": Vbar, "lambar": lambar}
    A = _matrices(case["kind"], n, 1, seed)[0]
    if op == "psd":
        return {"case": case, "A": A.float()}
    if op == "grad":
        g = torch.Generator(device="cuda")
        g.manual_seed(seed + 1)
        return {"case": case, "A": A, "w": torch.randn(n, generator=g, device="cuda", dtype=torch.float64),
                "B": torch.randn((n, 16), generator=g, device="cuda", dtype=torch.float64)}
    if op == "values":
        A = A.to(DTYPE[case["dtype"]])
    return {"case": case, "A": A}


def _signed(V):
    """Columns whose components sum to a non-negative value."""
    return V * torch.where(V.sum(-2, keepdim=True) < 0, -1.0, 1.0).to(V.dtype)


def run(state):
    case = state["case"]
    op, n = case["op"], case["n"]
    if op == "solve":
        lam, V = cv.symm_eig_solve(state["A"], bandwidth=case.get("b", 0), block=case.get("k", 0))
        return lam, _signed(V)
    if op == "psd":
        lam, V = cv.symm_eig_solve(state["A"])
        S = V.mT * lam.clamp(min=0).sqrt()[:, None]  # rows: scaled eigenvectors
        P = torch.empty_like(state["A"])
        cv.gemm(0, 1, n, n, n, 1.0, S, n, S, n, 0.0, P, n)
        return lam, P
    if op == "grad":
        A = state["A"].detach().requires_grad_()
        lam, V = autograd.eigh(A)
        loss = (state["w"] * lam).sum() + (V[:, :case["rank"]].mT @ state["B"]).square().sum()
        loss.backward()
        return loss.detach(), lam.detach(), A.grad
    if op == "values":
        return cv.symm_eig_values(state["A"], case["lo"], case["hi"])
    if op == "batched":
        lam, V = cv.symm_eig_batched(state["A"])
        return lam, _signed(V)
    if op == "sqrtm":
        lam, V = cv.symm_eig_batched(state["A"])
        S = V * lam.clamp(min=0).sqrt().sqrt()[:, None, :]
        return lam, torch.matmul(S, S.mT.contiguous())
    return cv.eig_backward(state["V"], state["lam"], state["Vbar"], state["lambar"])[0]


def exact(case, seed):
    op, n = case["op"], case["n"]
    if op != "backward" and n > 4100:
        return None  # a dense eigensolve of this size takes too long
    s = prepare(case, seed)
    if op == "solve":
        lam, V = torch.linalg.eigh(s["A"])
        return lam, _signed(V)
    if op == "psd":
        lam, V = torch.linalg.eigh(s["A"].double())
        return lam, (V * lam.clamp(min=0)) @ V.mT
    if op == "grad":
        k = case["rank"]
        lam, V = torch.linalg.eigh(s["A"])
        X = s["B"].mT @ V  # rows: B^T V
        loss = (s["w"] * lam).sum() + X[:, :k].square().sum()
        Vbar = torch.zeros_like(V)
        Vbar[:, :k] = 2.0 * (s["B"] @ X[:, :k])
        return loss, lam, _backward(V, lam, Vbar, s["w"])
    if op == "values":
        return torch.linalg.eigvalsh(s["A"].double())[case["lo"]:case["hi"] + 1]
    if op in ("batched", "sqrtm"):
        if case["batch"] > 4096:
            return None
        lam, V = torch.linalg.eigh(s["A"].double().cpu())
        lam, V = lam.cuda(), V.cuda()
        if op == "batched":
            return lam, _signed(V)
        return lam, torch.matmul(V * lam.clamp(min=0).sqrt()[:, None, :], V.mT.contiguous())
    return _backward(s["V"].double(), s["lam"].double(), s["Vbar"].double(), s["lambar"].double())


def _backward(V, lam, Vbar, lambar):
    C = V.mT @ Vbar
    gap = lam[None, :] - lam[:, None]
    gap.fill_diagonal_(1.0)
    K = 0.5 * (C - C.mT) / gap
    K.diagonal().copy_(lambar)
    return V @ K @ V.mT


def work(case):
    """Input read once and output written once; the reduction to tridiagonal form is
    4/3 n^3 flops, the transformation of n vectors 2 n^3, a dense product 2 n^3."""
    op, n = case["op"], case["n"]
    if op == "solve":
        return {"bytes": 8.0 * (2 * n * n + n), "flops": 10.0 / 3.0 * n ** 3}
    if op == "psd":
        return {"bytes": 4.0 * (2 * n * n + n), "flops": 13.0 / 3.0 * n ** 3}  # symmetric result
    if op == "grad":
        # the cotangent of V has rank-many non-zero columns: the products with it are thin
        return {"bytes": 8.0 * 2 * n * n, "flops": (10.0 / 3.0 + 3.0) * n ** 3}
    if op == "values":
        s = 8 if case["dtype"] == "f64" else 4
        return {"bytes": float(s) * (n * n + case["hi"] - case["lo"] + 1), "flops": 4.0 / 3.0 * n ** 3}
    if op in ("batched", "sqrtm"):
        s = 8 if op == "batched" else 4
        return {"bytes": float(s) * case["batch"] * (2 * n * n + n),
                "flops": case["batch"] * (10.0 / 3.0 + (1.0 if op == "sqrtm" else 0.0)) * n ** 3}
    return {"bytes": 4.0 * (3 * n * n + 2 * n), "flops": 5.0 * n ** 3}  # symmetric result
