"""CPU check of the tile lists that the coarse solve's triangular products read
(csrc/coarse_schedule.cpp), with tests/native/tile_lists_check.cpp."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = [os.path.join(ROOT, "tests", "native", "tile_lists_check.cpp"),
       os.path.join(ROOT, "topopt-in-openmp-gpu_amd", "csrc", "coarse_schedule.cpp")]


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("lists") / "tile_lists_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-o", exe] + SRC, check=True)
    return exe


@pytest.mark.parametrize("n,bw,planes", [
    (17 * 243, 0, 17),   # coarse 16x8x8, 4 tiles per plane
    (13 * 147, 0, 13),   # 3 tiles per plane
    (2 * 48, 0, 2),
    (300 * 12, 0, 300),  # many small planes
    (700, 150, 0),       # banded
    (64, 63, 0),
])
def test_lists_are_the_reach(checker, n, bw, planes):
    out = subprocess.run([checker, str(n), str(bw), str(planes)], capture_output=True, text=True,
                         timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.stdout + out.stderr
