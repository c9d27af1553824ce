"""The kernel that stages 3x3 layers' input in LDS run on the CPU (tests/cpp/staged_check.cpp): where it reads and writes."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = "/opt/rocm/lib/llvm/bin/clang++"   # the device code's vector types and half values need a compiler that has them


@pytest.mark.skipif(not os.path.exists(CLANG), reason="needs ROCm's clang++")
def test_every_form_stays_inside_its_operands(tmp_path):
    exe, cpp = str(tmp_path / "staged_check"), os.path.join(ROOT, "tests", "cpp")
    subprocess.check_call([CLANG, "-x", "c++", "-std=c++17", "-O1", "-ffp-contract=off", "-w", "-I" + os.path.join(cpp, "host_kernels"),
                           os.path.join(cpp, "staged_check.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
