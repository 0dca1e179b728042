"""The host side of the C entry points without a GPU: the library against a
stand-in for the HIP runtime on host memory (tests/native/fake_hip.hpp), a
child process per check of tests/native/host_calls_check.cpp."""
import os
import shutil
import subprocess

import pytest

import top3d_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    top3d_amd.library()
    lib = os.path.join(ROOT, "topopt-in-openmp-gpu_amd", "lib")
    exe = str(tmp_path_factory.mktemp("host") / "host_calls_check")
    subprocess.run([gxx, "-O1", "-std=c++17", "-rdynamic", "-o", exe,
                    os.path.join(ROOT, "tests", "native", "host_calls_check.cpp"),
                    "-L" + lib, "-ltop3d_hip", "-Wl,-rpath," + lib,
                    f"-Wl,-rpath-link,{ROCM}/lib", "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("check", ["filter_sums", "filter_without_memory",
                                   "change_without_memory", "given_back", "shapes_by_device",
                                   "sweep_timing"])
def test_host_calls(checker, check):
    out = subprocess.run([checker, check], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "OK", out.stdout + out.stderr
