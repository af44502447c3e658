"""Which eigenvalue kernel takes a batch (linalg.h): the faster one where the
two, timed apart, differ, over sizes 1 to 40 and batches
from 33 to 200000; never the wavefront kernel above 64 rows."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def by_wave(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("eig") / "eig_rule")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host", "eig_rule.cpp"), "-o", exe], check=True, timeout=300)
    return lambda batch, n: subprocess.run([exe, str(batch), str(n)], capture_output=True, text=True,
                                           check=True, timeout=60).stdout.strip() == "1"


@pytest.mark.parametrize("n,batch,wave", [
    (1, 9000, True), (1, 24000, True), (1, 200000, False), (2, 9000, True), (3, 6000, True), (3, 12000, False), (5, 12000, False), (2, 33, True), (2, 46000, False), (4, 514, True), (4, 2000, True),
    (4, 20000, False), (6, 6000, True), (6, 46000, False), (9, 514, True), (9, 6000, True), (9, 9000, True), (9, 12000, False),
    (9, 48000, False), (13, 9000, True), (13, 48000, False), (16, 130, True), (16, 9000, True), (16, 12000, True), (16, 24000, False),
    (20, 12000, True), (20, 16000, True), (20, 24000, False), (25, 24000, True), (25, 48000, False), (32, 12000, True), (40, 24000, True), (64, 514, True),
    (65, 2, False)])
def test_faster_kernel(by_wave, n, batch, wave):
    assert by_wave(batch, n) == wave
