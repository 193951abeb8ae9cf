"""A step whose allocations fail (tests/memory_caller.cpp refuses them from the host): the call reports
it, and the next call, which has the memory, gives the same density as if nothing had happened.
"""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from test_gpu_nonrect import _box_scene

pytestmark = pytest.mark.gpu

PKG_DIR = os.path.join(ROOT, "flux-interpolated-advection_amd")
SHAPE, CFL, H = (36, 40, 40), 4.0, 1.0 / 64


@pytest.fixture(scope="module")
def run(fia, scenes, tmp_path_factory):
    if fia.device_count() < 1:
        pytest.skip("no GPU visible")
    d = tmp_path_factory.mktemp("memory")
    exe = str(d / "memory_caller")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(ROOT, "tests", "memory_caller.cpp"), "-L", PKG_DIR, "-lfia", "-ldl",
                    "-Wl,-rpath," + PKG_DIR, "-o", exe], check=True, capture_output=True, text=True)
    fields = _box_scene(scenes, SHAPE, 11, CFL, H)
    for name, a in zip(("rho", "u", "v", "w"), fields):
        a.astype(np.float32).tofile(str(d / (name + ".bin")))
    r = subprocess.run([exe, str(d)] + [str(n) for n in SHAPE] + [repr(H), repr(float(fields[4]))], capture_output=True,
                       text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0
    rows = {}
    for line in r.stdout.splitlines():
        t = line.split()
        if t[0] == "deny":
            rows[int(t[1])] = {"refused": int(t[3]), "status": int(t[5]), "bytes": int(t[7]), "again": int(t[9])}
        elif t[0] == "asked":
            rows["asked"] = [int(x) for x in t[1:]]
        elif t[0] == "free":
            rows["free"] = {"status": int(t[1]), "bytes": int(t[3])}
    return d, rows, fields


def _density(d, name):
    return np.fromfile(str(d / (name + ".bin")), dtype=np.float32).reshape(SHAPE)


def test_failed_allocation_leaves_no_error(run):
    print("case refused allocations", flush=True)
    d, rows, _ = run
    failed = [s for s in rows if isinstance(s, int) and rows[s]["status"] != 0]
    assert len(failed) > 5   # the scratch that a step needs
    for s in failed:
        assert rows[s]["status"] == 5 and rows[s]["again"] == 0
        assert np.array_equal(_density(d, "again_%d" % s), _density(d, "free"))
