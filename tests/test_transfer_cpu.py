"""The library's runtime on a host-side stand-in for the HIP runtime (tests/cpp/host_device.hip): what several
threads that share a context may expect of them, without a GPU."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    """Runs a check of tests/cpp/transfer_check.hip against the library's sources, compiled for the host alone."""
    tmp = tmp_path_factory.mktemp("transfer")
    sources = [os.path.join(ROOT, "excalibur_amd", "csrc", f) for f in ("transfer.hip", "runtime.hip")]
    sources += [os.path.join(ROOT, "tests", "cpp", f) for f in ("host_device.hip", "transfer_check.hip")]
    objects = [str(tmp / (os.path.basename(s) + ".o")) for s in sources]

    def build(pair):
        subprocess.check_call([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-fuse-cuid=none", "-O1", "-fPIC", "-std=c++17", "-c", pair[0], "-o", pair[1]])

    with ThreadPoolExecutor() as pool:
        list(pool.map(build, zip(sources, objects)))
    exe = str(tmp / "transfer_check")
    subprocess.check_call(["g++", "-pthread", "-Wl,--allow-multiple-definition", "-rdynamic", "-o", exe] + objects + ["-ldl"])

    def run(name):
        out = subprocess.run([exe, name], capture_output=True, text=True, timeout=120)
        assert out.returncode == 0, out.stdout[-2000:] + out.stderr

    return run


def test_threads_that_share_a_context_get_one_split_scratch(check):
    check("scratch")


def test_threads_that_share_a_context_copy_at_once(check):
    check("shared")


def test_helper_threads_sleep_while_the_link_works(check):
    check("idle")


def test_a_process_at_its_thread_limit_copies_without_helpers(check):
    check("limit")
