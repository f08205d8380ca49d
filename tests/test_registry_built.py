"""Names of the kernels as the built library registers them, whatever macros
they come from: unique within the line / column form (the tuning cache, a
chosen stage kernel and the packed twins are found by name), with every kind
present."""
import collections
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "2decomp-fft_amd")
ROCM = "/opt/rocm"


@pytest.fixture(scope="module")
def names(d2d, tmp_path_factory):
    d2d.lib()
    if not shutil.which("g++") or not os.path.exists(ROCM + "/include/hip/hip_runtime.h"):
        pytest.skip("g++ or the HIP headers not found")
    exe = str(tmp_path_factory.mktemp("host") / "registry_names")
    r = subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM + "/include",
                        "-I" + ROOT + "/include", "-I" + os.path.join(PKG, "csrc"),
                        os.path.join(ROOT, "tests", "host", "registry_names.cpp"), "-L" + PKG, "-ld2dhip",
                        "-L" + ROCM + "/lib", "-lamdhip64", "-Wl,-rpath," + PKG, "-Wl,-rpath," + ROCM + "/lib",
                        "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    return [tuple(line.split(" ", 1)) for line in out.splitlines()]


def test_names_unique(names):
    dup = [k for k, c in collections.Counter(names).items() if c > 1]
    assert not dup, dup


def test_every_kind_is_registered(names):
    have = {n for _, n in names}
    kinds = collections.Counter(n.split()[4] for n in have if n.split()[0] in ("double", "float") and "mixed" not in n)
    for k in ("c2c", "r2c", "c2r", "dct2", "dct3", "dctx", "dct4", "ypk", "yun", "yup"):
        assert kinds[k] >= 9, (k, kinds)
    for t in ("double", "float"):
        for tag in ("", " primes", " chirp"):
            for k in ("c2c", "r2c", "c2r", "dct"):
                name = "%s mixed %s%s" % (t, k, tag)
                assert {("0", name), ("1", name)} <= set(names), name
    assert any(n.startswith("mfma") for n in have)
