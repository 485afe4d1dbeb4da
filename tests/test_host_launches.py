"""The library's host side against a HIP runtime that runs no kernel and checks
each launch against what its function was granted (host_runtime/launches.cpp):
faults that one GPU, or one grid alive at a time, does not show."""
import os
import subprocess

import pytest

from fluid_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    if not os.path.exists(build.LIB):
        build.build()
    exe = str(tmp_path_factory.mktemp("host_runtime") / "launches")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(build.ROOT, "include"), "-rdynamic",
                    os.path.join(HERE, "host_runtime", "launches.cpp"), "-o", exe, "-ldl"], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["cm11a_bytes", "cm11a_two_grids", "extrapolate_bytes", "two_devices"])
def test_host_side(launches, scenario):
    r = subprocess.run([launches, build.LIB, scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
