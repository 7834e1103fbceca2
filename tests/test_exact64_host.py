"""The FP64 flux functions that share the reciprocals of a denominator
(kr_exact64.h), compiled for the host, against the general functions bit for
bit over the whole range of their guard: transverse velocities and fields of
0, of ordinary size, at the guard's limit and down to the smallest subnormals,
states that differ by ulps, units far from 1."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "kratos_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("exact64")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text("")
    exe = d / "exact64_host"
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-w", f"-I{d}", f"-I{CSRC}",
                    os.path.join(HERE, "exact64_host.cpp"), "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("low", [-1073, -1030, -900, -842, -838, -500])
def test_equals_general_functions(program, low):
    n = 200000
    out = subprocess.run([str(program), str(n), str(low)], check=True, capture_output=True, text=True).stdout
    for line in out.splitlines():
        in_range, bad = map(int, line.split())
        assert in_range > 0.9 * n
        assert bad == 0
