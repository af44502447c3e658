"""The staged copies between the caller's arrays and the device on the CPU
(tests/host/transfer_check.cpp): the library's transfer unit with a model of
the runtime whose copies run as late as they may, around the size where staging
begins, without threads, with a failing copy, and in the background."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pyrpa_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("transfer") / "transfer_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host", "transfer_check.cpp"), "-x", "c++", os.path.join(CSRC, "transfer.hip"),
                    "-o", exe, "-pthread", "-ldl", "-rdynamic"], check=True, timeout=300)
    return exe


@pytest.mark.parametrize("what", ["sizes", "no_threads", "release", "failed_copy", "background"])
def test_staged_copies(check, what):
    r = subprocess.run([check, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
