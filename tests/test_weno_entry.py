"""The z stencils' interpolants of the quadrature tables (csrc/fia_math.hpp weno6_entry), built for
the host, against WENO6 in numpy FP64 (Newton-form candidates, ideal weights, smoothness
indicators in the samples' differences), for both weight forms.

Tolerance: with M the largest |sample|, the evaluated terms are at most t |g_2| + |t (t - 1) Q / D|
<= 2 M + 2 M (1 + 4 / 7.5 + 1 / 15) / 0.53 < 8 M, in about ten FP32 operations and coefficients of
relative rounding 2^-24: 10 * 8 * 2^-24 M < 5e-6 M.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FORMS = ((244, -683, 634), (244, -293, 244), (634, -683, 244))


@pytest.fixture(scope="module")
def entry(tmp_path_factory):
    hipcc = "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    out = str(tmp_path_factory.mktemp("entry") / "weno_entry_host.so")
    subprocess.run([hipcc, "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(ROOT, "tests", "weno_entry_host.cpp"), "-o", out],
                   check=True, capture_output=True)
    L = ctypes.CDLL(out)
    L.host_entry_value.argtypes = [ctypes.POINTER(ctypes.c_double), ctypes.c_double, ctypes.c_double, ctypes.c_int]
    L.host_entry_value.restype = ctypes.c_double
    return L


def _reference(f, t, kappa, opt):
    d = [t + 2 - i for i in range(6)]
    c = (d[4] * d[5] / 20, -d[5] * d[0] / 10, d[0] * d[1] / 20)
    num = den = 0.0
    for r in range(3):
        p, x = f[r:r + 4], d[r]
        value = (p[0] + x * (p[1] - p[0]) + x * (x - 1) / 2 * (p[2] - 2 * p[1] + p[0])
                 + x * (x - 1) * (x - 2) / 6 * (p[3] - 3 * p[2] + 3 * p[1] - p[0]))
        a, b = p[2] - 2 * p[1] + p[0], p[3] - 2 * p[2] + p[1]
        k = FORMS[r]
        s = kappa / 180 * (180 * (f[3] - f[2]) ** 2 + k[0] * a * a + k[1] * a * b + k[2] * b * b)
        w = c[r] / (1e-30 + s * s) if opt else c[r] / (1e-6 + s) ** 2
        num, den = num + w * value, den + w
    return num / den


@pytest.mark.parametrize("opt", [False, True])
@pytest.mark.parametrize("kappa", [1.0, 1.0 / 64 ** 2, 1.0 / 256 ** 2])
@pytest.mark.parametrize("scale,step", [(1.0, False), (1.0, True), (3e-4, False), (250.0, True), (0.0, False)])
def test_entry_matches_weno6(entry, opt, kappa, scale, step):
    rng = np.random.default_rng(5)
    for _ in range(300):
        f = rng.uniform(-1, 1, size=6) if not step else np.where(np.arange(6) < rng.integers(1, 6), 1.0, rng.uniform(-1, 0.9))
        f = (scale * f).astype(np.float32).astype(np.float64)
        for t in (0.0, float(np.float32(rng.uniform())), 0.5, 1.0):
            got = entry.host_entry_value(f.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), t, kappa, int(opt))
            assert abs(got - _reference(f, t, kappa, opt)) <= 5e-6 * np.abs(f).max(), (f, t)


@pytest.mark.parametrize("mz", [1, 2, 3, 7, 64])
def test_entry_index_covers_every_clamped_stencil(entry, mz):
    # a base past the row's entries has the same clamped samples as the entry it takes
    last = mz + entry.host_entry_pad() - 1
    for base in list(range(-9, mz + 9)) + [-(1 << 24), 1 << 24]:
        e = entry.host_entry_index(base, mz)
        assert 0 <= e <= last
        clamp = lambda b: [min(max(b - 2 + i, 0), mz - 1) for i in range(6)]
        assert clamp(base) == clamp(e - 3)
