"""Admission of concurrent solves: which persistent grids may be on the GPU together (host code, in a
C++ program of its own)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_admission(tmp_path):
    exe = str(tmp_path / "residency_test")
    p = subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall", os.path.join(ROOT, "tests", "cpp", "residency_test.cpp"),
                        "-o", exe], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and "residency ok" in p.stdout, p.stdout
