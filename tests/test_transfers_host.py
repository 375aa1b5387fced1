"""Host code of the transfers without a GPU: executor.cpp and xfer.cpp built with the host compiler against a runtime of
host memory (tests/native/host_runtime.cpp), which runs a stream's work on a thread of its own and can make allocations,
copies and waits fail."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "splatx-metal_amd", "csrc")
HIP = "/opt/rocm/include"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(HIP), reason="needs g++ and the HIP headers")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("transfers") / "transfers")
    native = os.path.join(REPO, "tests", "native")
    src = [os.path.join(native, "transfers.cpp"), os.path.join(native, "host_runtime.cpp"),
           os.path.join(CSRC, "executor.cpp"), os.path.join(CSRC, "xfer.cpp")]
    # (the steps' kernels are not linked: nothing here calls them)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-I", HIP, "-I", os.path.join(REPO, "include"),
                    "-I", CSRC, *src, "-o", exe, "-pthread", "-Wl,--unresolved-symbols=ignore-all"], check=True)
    return exe


@pytest.mark.parametrize("check", ["upload_fails_midway", "error_is_reported_once", "without_the_ring", "kept_memory_gives_way",
                                   "kept_memory_follows_use", "several_threads"])
def test_transfers(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
