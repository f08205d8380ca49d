"""The planner of the kernels of any length (csrc/mixed_plan.cpp), on the CPU:
a length that a kernel says it runs has a launch shape within its limits (a
plan fails where it has none), over all lengths, element sizes, transform
kinds and both forms; the lengths whose best schedule needs more rows than a
workgroup has threads run on another schedule."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "2decomp-fft_amd")
ROCM = "/opt/rocm"
IO = {"c2c": 0, "r2c": 1, "c2r": 2, "r2r": 3}


@pytest.fixture(scope="module")
def shapes(d2d, tmp_path_factory):
    d2d.lib()
    if not shutil.which("g++") or not os.path.exists(ROCM + "/include/hip/hip_runtime.h"):
        pytest.skip("g++ or the HIP headers not found")
    exe = str(tmp_path_factory.mktemp("host") / "mixed_shapes")
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM + "/include",
                        "-I" + ROOT + "/include", "-I" + os.path.join(PKG, "csrc"),
                        os.path.join(ROOT, "tests", "host", "mixed_shapes.cpp"), "-L" + PKG, "-ld2dhip",
                        "-L" + ROCM + "/lib", "-lamdhip64", "-Wl,-rpath," + PKG, "-Wl,-rpath," + ROCM + "/lib",
                        "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]

    def run(*args):
        q = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True, timeout=300)
        assert q.returncode == 0, q.stderr[-2000:]
        return q.stdout.splitlines()
    return run


def test_every_length_that_runs_has_a_shape(shapes):
    out = shapes()
    assert out[:-1] == []
    assert int(out[-1].split()[1]) > 100000


@pytest.mark.parametrize("rb,io,lines,n", [
    (8, "c2c", 0, 6125), (8, "c2c", 1, 6125), (8, "r2c", 1, 6125), (8, "c2r", 0, 6125), (4, "c2c", 1, 6125),
    (4, "c2c", 0, 6125), (8, "r2r", 0, 5250), (8, "r2r", 1, 5250), (4, "r2r", 1, 5250), (8, "r2r", 1, 6125),
    (8, "c2c", 0, 6000), (8, "c2c", 1, 6144)])
def test_longest_lengths_run(shapes, rb, io, lines, n):
    """Lengths near the six points per thread of a full workgroup."""
    assert len(shapes(rb, IO[io], lines, n)) == 1
