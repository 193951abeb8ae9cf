"""The forms that the flux passes' launchers choose by size and rule, on the CPU (tests/forms_host.cpp)."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT


def build_forms(out, sanitize=False):
    cmd = ["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-std=c++17", "-fPIC", "-shared",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I/opt/rocm/include", os.path.join(ROOT, "tests", "forms_host.cpp"), "-o", out]
    if sanitize:
        cmd[5:5] = ["-Xarch_host", "-fsanitize=address", "-fno-omit-frame-pointer"]
    subprocess.run(cmd, check=True, capture_output=True)
    return out


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    if not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("hipcc not found")
    L = ctypes.CDLL(build_forms(str(tmp_path_factory.mktemp("forms") / "forms_host.so")))
    L.forms_zero_chunk.argtypes = [ctypes.c_int] * 4
    L.forms_zero_chunk.restype = ctypes.c_long
    return L


def test_zero_velocity_march_fits_a_launch(forms):
    # gridDim.y holds at most 65,535 chunks, also of a box of millions of planes; the planes per thread
    # of ordinary grids stay those that were measured
    for shape, chunk in (((256, 256, 256), 32), ((128, 128, 128), 8), ((75, 96, 50), 4), ((32, 32, 32), 1)):
        assert forms.forms_zero_chunk(*shape, 256) == chunk
    for nx in (1, 7, 65535, 65536, 2097120, 2097121, 3000000, 50000000):
        for block in (64, 128, 256):
            chunk = forms.forms_zero_chunk(nx, 3, 4, block)
            assert 1 <= chunk and -(-nx // chunk) <= 65535
