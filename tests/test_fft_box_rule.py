"""Which box size a pass takes (fftbox.h) against the times of both, each pass
timed alone: whole boxes where the quarter-size ones need a second round, small
ones where they all run at once, whole ones on a full chip."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "pyrpa_amd")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def passes(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rule") / "fft_rule")
    subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-host-only", "-x", "hip", "-c",
                    os.path.join(HERE, "host", "fft_rule.cpp"), "-o", exe + ".o"], check=True, timeout=300)
    subprocess.run([HIPCC, exe + ".o", os.path.join(PKG, "libgmod.so"), "-Wl,-rpath," + PKG, "-o", exe], check=True,
                   timeout=300)
    return lambda *a: subprocess.run([exe, *map(str, a)], capture_output=True, text=True, check=True,
                                     timeout=60).stdout.strip()


@pytest.mark.parametrize("prec,dims,mask,n,want", [
    (0, (32, 32, 1, 512), 7, 1, "s"), (0, (32, 32, 1, 512), 8, 1, "s"), (0, (16, 16, 8, 256), 8, 1, "s"),
    (0, (64, 64, 1, 256), 7, 1, "s"), (1, (32, 32, 1, 1024), 7, 1, "s"), (1, (16, 16, 16, 256), 8, 1, "s"),
    (0, (40, 32, 1, 512), 7, 1, "s"), (1, (48, 48, 1, 512), 7, 1, "s"),  # the quarter box is not tiled: two a CU
    (0, (48, 32, 1, 512), 7, 1, "w"), (0, (16, 16, 8, 512), 7, 1, "w"), (0, (16, 16, 8, 512), 8, 1, "w"),
    (0, (64, 48, 1, 512), 8, 1, "w"), (0, (16, 16, 1, 4096), 7, 1, "w"), (1, (32, 32, 4, 512), 15, 1, "ww"),
    (1, (96, 32, 1, 512), 7, 1, "w"), (1, (64, 64, 1, 512), 8, 1, "w"),
    (0, (16, 16, 4, 256), 15, 2, "ss"), (0, (16, 16, 4, 256), 15, 4, "ww"), (0, (32, 32, 1, 2048), 15, 1, "ww"),
    (0, (32, 32, 16, 2048), 15, 1, "www")])
def test_tiled_passes(passes, prec, dims, mask, n, want):
    assert passes(prec, *dims, mask, n) == want


@pytest.mark.parametrize("prec,dims,mask,n,want", [
    (1, (18, 18, 1, 90), 7, 1, "s"), (1, (18, 14, 1, 150), 8, 1, "s"), (0, (48, 48, 12, 150), 8, 1, "s"),
    (1, (80, 80, 4, 240), 8, 1, "s"), (0, (100, 100, 3, 720), 7, 1, "sss"), (0, (128, 128, 1, 1000), 1, 1, "W"), (0, (27, 27, 5, 180), 15, 9, "ss"),
    (1, (24, 24, 6, 200), 15, 21, "ws"), (1, (24, 24, 6, 200), 15, 15, "ws"), (0, (50, 64, 4, 300), 8, 1, "W"),
    (1, (36, 36, 5, 288), 8, 1, "W"), (0, (30, 30, 12, 140), 7, 1, "WW"), (1, (45, 32, 1, 4096), 7, 1, "W"),
    (1, (24, 45, 6, 2400), 8, 1, "W"), (0, (80, 80, 1, 1250), 7, 1, "W"), (1, (50, 15, 1, 800), 8, 1, "W"),
    (1, (25, 25, 6, 800), 8, 1, "w")])  # a capital: one box a CU
def test_untiled_passes(passes, prec, dims, mask, n, want):
    assert passes(prec, *dims, mask, n) == want
