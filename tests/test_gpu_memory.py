"""Scratch that a step can do without, on a device that has no memory for it (tests/memory_caller.cpp
refuses allocations from the host): the z stencil tables of the WENO6 integral quadrature, the twisted
faces' fixed records and the piece records' room to grow.  The step must take the form that needs
less, agree with the oracle at the density step's bar, and leave no error behind; an allocation that
it cannot do without must find the memory that idle tables hold, on its own context or another.
"""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, rel_linf
from test_gpu_nonrect import _box_scene

pytestmark = pytest.mark.gpu

PKG_DIR = os.path.join(ROOT, "flux-interpolated-advection_amd")
TOL = 1e-5
SHAPE, CFL, H = (36, 40, 40), 4.0, 1.0 / 64      # 135 bricks: the tables are taken


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
            rows["deny", t[1]] = {"refused": int(t[3]), "status": int(t[5]), "bytes": int(t[7]), "again": int(t[9])}
        elif t[0] == "asked":
            rows["asked"] = [int(x) for x in t[1:]]
        elif t[0] == "free":
            rows["free"] = {"status": int(t[1]), "bytes": int(t[3])}
        elif t[0][:4] in ("one_", "two_"):
            rows[t[0]] = {"status": (int(t[1]), int(t[2])), "bytes": (int(t[4]), int(t[5])), "refused": int(t[9])}
    return d, rows, fields


def _density(d, name):
    return np.fromfile(str(d / (name + ".bin")), dtype=np.float32).reshape(SHAPE)


def _runs_of_five(sizes):
    """The sizes asked for five times in a row, in order: the piece records, then the fixed ones."""
    return [s for i, s in enumerate(sizes[:-4]) if all(x == s for x in sizes[i:i + 5]) and (i == 0 or sizes[i - 1] != s)]


def _tables():
    nx, ny, nz = SHAPE
    return [32 * (nz + 5) * nx * ny, 32 * (nz + 5) * nx * (ny + 1)]


@pytest.fixture(scope="module")
def reference(oracle, run):
    rho, u, v, w, dt = run[2]
    return oracle.move_substances(rho.astype(np.float64), u, v, w, H, dt, split="xz-CellFaceAligned")


def test_step_without_tables_matches_oracle(run, reference):
    print("case no memory for the tables", flush=True)
    d, rows, _ = run
    assert rows["free"]["status"] == 0 and set(_tables()) <= set(rows["asked"])
    assert rel_linf(_density(d, "free"), reference) < TOL
    for s in _tables():
        r = rows["deny", str(s)]
        assert r["refused"] > 0 and r["status"] == 0 and r["again"] == 0
        assert r["bytes"] == rows["free"]["bytes"] - sum(_tables())
        assert rel_linf(_density(d, "deny_%d" % s), reference) < TOL
        assert np.array_equal(_density(d, "again_%d" % s), _density(d, "free"))


def test_step_without_room_to_grow_is_the_same(run):
    print("case no memory for more than the records", flush=True)
    d, rows, _ = run
    records = _runs_of_five(rows["asked"])
    assert len(records) >= 2   # piece records, and the fixed records of the twisted faces
    # the fixed records not even exactly: the pieces are counted, cut and summed in the same order
    for name in ["%d" % s for s in records[:2]] + ["%d_exact" % records[1]]:
        r = rows["deny", name]
        assert r["refused"] > 0 and r["status"] == 0 and r["again"] == 0
        assert np.array_equal(_density(d, "deny_" + name), _density(d, "free"))


def test_failed_allocation_leaves_no_error(run):
    print("case refused allocations", flush=True)
    d, rows, _ = run
    failed = [k for k, r in rows.items() if k[0] == "deny" and r["status"] != 0]
    assert len(failed) > 5   # the scratch that a step needs
    for k in failed:
        assert rows[k]["status"] == 5 and rows[k]["again"] == 0
        assert np.array_equal(_density(d, "again_" + k[1]), _density(d, "free"))


@pytest.mark.parametrize("contexts", ["one", "two"])
def test_tables_are_given_back_for_scratch_that_is_needed(run, reference, contexts):
    print("case tables given back", contexts, flush=True)
    d, rows, _ = run
    lean, capped = rows[contexts + "_lean"], rows[contexts + "_capped"]
    assert lean["status"] == (0, 0) and capped["status"] == (0, 0)
    assert capped["refused"] > 0
    for name in (contexts + "_lean", contexts + "_capped"):
        assert rel_linf(_density(d, name), reference) < TOL
        assert np.array_equal(_density(d, name + "_p"), _density(d, "one_lean_p"))
