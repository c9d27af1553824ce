"""Kernels on slices of wider tensors, run on the CPU with every tensor ending at an unreadable page (tests/cpp/slices_check.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = "/opt/rocm/lib/llvm/bin/clang++"   # the device code's vector types and half values need a compiler that has them


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs ROCm's clang++")
def test_slices_are_read_and_written_inside_their_tensors(tmp_path):
    exe, cpp = str(tmp_path / "slices_check"), os.path.join(ROOT, "tests", "cpp")
    subprocess.check_call([CLANG, "-x", "c++", "-std=c++17", "-O0", "-ffp-contract=off", "-w", "-I" + os.path.join(cpp, "host_kernels"),
                           os.path.join(cpp, "slices_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
