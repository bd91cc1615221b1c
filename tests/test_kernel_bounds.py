"""Every access of the four-kernel path inside its arrays: the kernels compiled as host code under
AddressSanitizer (tests/host_kernels), a right-hand side and two Runge-Kutta stages at every degree. Degrees whose
node count does not fill whole waves have lanes without a node, which must stay away from the arrays. At
N = 1 these are 56 of 64 lanes."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "flexi_amd", "csrc")


@pytest.fixture(scope="module")
def four_kernels(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    src = os.path.join(HERE, "host_kernels")
    exe = str(tmp_path_factory.mktemp("host_kernels") / "four_kernels")
    r = subprocess.run([cxx, "-std=c++20", "-O0", "-w", "-fsanitize=address", "-pthread", "-I", src, "-I", CSRC,
                        os.path.join(src, "four_kernels.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return exe


@pytest.mark.parametrize("N", range(1, 8))
def test_four_kernels_stay_in_their_arrays(four_kernels, N):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([four_kernels, str(N)], capture_output=True, text=True, env=env, timeout=120)
    # (the report names the kernel and the array)
    assert r.returncode == 0, r.stdout[-200:] + r.stderr[:300] + r.stderr[r.stderr.find("is located"):][:400]
