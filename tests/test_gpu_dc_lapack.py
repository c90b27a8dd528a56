"""The device divide and conquer needs host LAPACK for leaves of more than 64 rows only."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import torch
import cuev_amd as cv
assert cv.lapack_name().endswith("libstub.so"), cv.lapack_name()
for dt, u in ((torch.float64, 2.3e-16), (torch.float32, 1.2e-7)):
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    n = 200
    G = torch.randn((n, n), generator=g, device="cuda", dtype=dt)
    A = (G + G.T) / 2
    lam, V = cv.symm_eig_solve(A)
    ref = torch.linalg.eigvalsh(A.cpu().double()).cuda()
    # backward error of the solve: at most about n roundings of ||A||
    assert float((lam.double() - ref).abs().max()) <= n * u * float(ref.abs().max())
    try:
        cv.symm_eig_solve(A, dc_mode="device", dc_leaf=100)
        raise SystemExit("leaves of 100 rows were solved without ?steqr")
    except cv.CuevError as e:
        assert e.name == "LAPACK_UNAVAILABLE", e
print("child ok")
"""


def test_default_leaves_without_steqr(tmp_path, torch_dev):
    """A LAPACK library that lacks ?steqr (its ?stedc is never called here)."""
    src, so = tmp_path / "stub.c", tmp_path / "libstub.so"
    src.write_text("void dstedc_(void) {}\nvoid sstedc_(void) {}\n")
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    env = dict(os.environ, CUEV_LAPACK_LIB=str(so), PYTHONPATH=ROOT)
    p = subprocess.run([sys.executable, "-c", CHILD], capture_output=True, text=True, timeout=100, env=env, cwd=ROOT)
    assert p.returncode == 0 and "child ok" in p.stdout, (p.stdout, p.stderr)
