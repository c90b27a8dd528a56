"""Device buffers kept between calls: sizes and order of their allocations (host code, in a C++ program
with a stand-in for the HIP allocator)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_allocations(tmp_path):
    exe = str(tmp_path / "idle_buffers_test")
    p = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                        os.path.join(ROOT, "tests", "cpp", "idle_buffers_test.cpp"),
                        os.path.join(ROOT, "cuev_amd", "csrc", "idle_buffers.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and "idle buffers ok" in p.stdout, p.stdout
