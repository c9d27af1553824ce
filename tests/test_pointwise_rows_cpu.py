"""The pointwise kernels' addressing of shortcuts and results, walked over shapes on the CPU with the header the kernels use."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pointwise_accesses_stay_inside_their_tensors(tmp_path):
    exe = str(tmp_path / "pw_rows_check")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-o", exe, os.path.join(ROOT, "tests", "cpp", "pw_rows_check.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
