"""A mesh read into a buffer that begins in pinned host memory and runs past its end is not
written through the pinned mapping (tests/cpp/readback_check.cpp: the read-back's host code on the
CPU, the HIP calls it makes replaced)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_read_back_keeps_to_pinned_allocations(tmp_path):
    exe = str(tmp_path / "readback_check")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", exe, os.path.join(ROOT, "tests", "cpp", "readback_check.cpp"),
                    os.path.join(ROOT, "leven_amd", "csrc", "lvn_readback.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
