"""The forms that the flux passes' launchers choose by size and rule, replayed on the CPU (tests/forms_host.cpp,
the kernels' own __host__ __device__ code) against the FP64 oracle and against the general forms.

Every field, psi and table lies between NaN guards in memory that starts as NaN, so these are also
checks of the index arithmetic: tiles of vertices, chunks of planes, table rows and clamped entries,
the box of a brick, fixed records.  They pin which form the GPU tests' scenes take: pieces that leave the
staged box, and twisted faces with more pieces than the fixed records hold.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, rel_linf
from test_gpu_nonrect import _box_scene
from test_pass_host import PSI, SPLIT, rel_linf_either, white_noise_scene

TOL = 1e-5
INTERP = {"linear": 0, "WENO6": 1, "1Dy_linear": 2, "1Dy_WENO6": 3, "WENO6-optimized": 4}
NONE, ALWAYS, RULE = -1, 1, 0      # the z stencil tables


def build_forms(out, sanitize=False):
    cmd = ["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", "-fPIC", "-shared",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I/opt/rocm/include", os.path.join(ROOT, "tests", "forms_host.cpp"), "-o", out]
    if sanitize:
        cmd[5:5] = ["-Xarch_host", "-fsanitize=address", "-fno-omit-frame-pointer"]
    subprocess.run(cmd, check=True, capture_output=True)
    return out


class Forms:
    COLS = ("twisted", "degenerate", "slots", "gen_over", "tables", "box", "memory", "gen_max")

    def __init__(self, path):
        L = ctypes.CDLL(path)
        vp, i, d = ctypes.c_void_p, ctypes.c_int, ctypes.c_double
        fp, dp, ip = ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)
        L.forms_create.restype = vp
        L.forms_destroy.argtypes = [vp]
        L.forms_message.argtypes = [vp]
        L.forms_message.restype = ctypes.c_char_p
        L.forms_zero_chunk.argtypes = [i] * 4
        L.forms_zero_chunk.restype = ctypes.c_long
        L.forms_move_substances.argtypes = [vp, i, i, i, d, fp, fp, fp, fp, d, i, i, i, i, d, i, i, dp, i, ip]
        L.forms_advect_velocity.argtypes = [vp, i, i, i, d, fp, fp, fp, i, fp, d, i, i, i, i, i, dp, i, ip]
        L.forms_flux_pass.argtypes = [vp, i, i, i, i, d, fp, fp, fp, fp, d, i, i, i, i, i, i, d, i, i, dp, i, ip]
        L.forms_vertices.argtypes = [vp, i, i, i, i, fp, fp, fp, d, i, i, fp]
        assert L.forms_cols() == len(self.COLS)
        self.L = L

    def _call(self, fn, *args):
        """Runs fn(ctx, *args, stats); the passes' stats rows as dicts."""
        c = self.L.forms_create()
        try:
            st = np.zeros((16, len(self.COLS)))
            rows = ctypes.c_int(0)
            e = fn(c, *args, st.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 16, ctypes.byref(rows))
            assert e == 0, (e, self.L.forms_message(c).decode())
        finally:
            self.L.forms_destroy(c)
        return [dict(zip(self.COLS, r.astype(int))) for r in st[:rows.value]]

    @staticmethod
    def _p(a):
        return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))

    def move_substances(self, rho, u, v, w, h, dt, split="xz-CellFaceAligned", interp="WENO6", tables=RULE, min_area=1.0):
        q = rho.copy()
        p = self._p
        st = self._call(self.L.forms_move_substances, *rho.shape, h, p(q), p(u), p(v), p(w), dt, SPLIT[split],
                        INTERP[interp], 1, 1, min_area, tables, 0)
        return q, st

    def advect_velocity(self, u, v, w, comp, h, dt, interp="WENO6", tables=RULE):
        out = np.full_like((u, v, w)[comp], np.nan)
        p = self._p
        st = self._call(self.L.forms_advect_velocity, u.shape[0] - 1, u.shape[1], u.shape[2], h, p(u), p(v), p(w), comp,
                        p(out), dt, INTERP[interp], 1, 1, tables, 0)
        return out, st

    def flux_pass(self, q, u, v, w, h, dt, split, interp, psi, zero, integral, comp=-1, tables=RULE, zero_chunk=0):
        q = q.copy()
        p = self._p
        st = self._call(self.L.forms_flux_pass, comp, u.shape[0] - 1, u.shape[1], u.shape[2], h, p(q), p(u), p(v), p(w),
                        dt, SPLIT[split], INTERP[interp], PSI[psi], int(zero), int(integral), 1, 1.0, tables, zero_chunk)
        return q, st

    def vertices(self, u, v, w, comp, dt_over_h, each):
        n = [s + (a == comp) + 1 for a, s in enumerate((u.shape[0] - 1, u.shape[1], u.shape[2]))]
        out = np.full([3] + n, np.nan, dtype=np.float32)
        c = self.L.forms_create()
        try:
            p = self._p
            assert self.L.forms_vertices(c, comp, u.shape[0] - 1, u.shape[1], u.shape[2], p(u), p(v), p(w), dt_over_h,
                                         INTERP["WENO6"], int(each), p(out)) == 0
        finally:
            self.L.forms_destroy(c)
        return out


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    if not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("hipcc not found")
    path = os.environ.get("FIA_FORMS_HOST") or build_forms(str(tmp_path_factory.mktemp("forms") / "forms_host.so"))
    return Forms(path)


def test_zero_velocity_march_fits_a_launch(forms):
    # gridDim.y holds at most 65,535 chunks, also of a box of millions of planes; the planes per thread
    # of ordinary grids stay those that were measured
    chunk_of = forms.L.forms_zero_chunk
    for shape, chunk in (((256, 256, 256), 32), ((128, 128, 128), 8), ((75, 96, 50), 4), ((32, 32, 32), 1)):
        assert chunk_of(*shape, 256) == chunk
    for nx in (1, 7, 65535, 65536, 2097120, 2097121, 3000000, 50000000):
        for block in (64, 128, 256):
            chunk = chunk_of(nx, 3, 4, block)
            assert 1 <= chunk and -(-nx // chunk) <= 65535


def test_tables_fit_a_launch(forms):
    # a launch counts its threads in 32 bits: 768 a brick of 4 x 8 x 16 cells, and one per table entry
    takes = forms.L.forms_takes_tables
    assert takes(256, 256, 256) and takes(36, 40, 40) and takes(900, 900, 900) and takes(18000, 1, 18000)
    assert not takes(24, 24, 24)            # fewer than 128 bricks
    assert not takes(19500, 1, 19500)       # 4875 x 1 x 1219 bricks
    assert not takes(31000, 31000, 1)       # 961 million rows of six entries


@pytest.mark.parametrize("comp", [-1, 0, 1, 2])
@pytest.mark.parametrize("shape", [(9, 15, 15), (8, 16, 14), (4, 14, 16), (1, 2, 3), (23, 33, 18), (70, 3, 40)])
def test_vertex_tiles_give_each_vertex_its_value(forms, shape, comp):
    # the tiles' shared passes and a vertex's own run the same evaluations; bar: FP32 rounding of the
    # largest displacement, a few operations' worth
    rng = np.random.default_rng(17)
    fields = [np.cumsum(rng.normal(size=[s + (a == b) for b, s in enumerate(shape)]), axis=(a + 1) % 3).astype(np.float32)
              for a in range(3)]
    scale = 2.0 / max(np.abs(f).max() for f in fields)
    tiles, each = [forms.vertices(*fields, comp, scale, e) for e in (0, 1)]
    assert np.isfinite(tiles).all()
    assert np.abs(tiles - each).max() <= 2e-6 * 2.0


# the scenes of tests/test_gpu_brick.py: whole bricks and remainders, boxes thinner than a brick; the last
# three throw pieces out of the staged box
@pytest.mark.parametrize("interp", ["WENO6", "WENO6-optimized"])
@pytest.mark.parametrize("shape,cfl,outside", [((16, 32, 128), 1.0, False), ((17, 33, 81), 2.0, False), ((66, 9, 50), 3.0, True),
                                               ((5, 71, 131), 4.0, True), ((36, 40, 40), 4.0, True)])
def test_density_step_on_bricks(forms, oracle, scenes, shape, cfl, outside, interp):
    h = 1.0 / 64
    rho, u, v, w, dt = _box_scene(scenes, shape, 11, cfl, h)
    q, st = forms.move_substances(rho, u, v, w, h, dt, interp=interp)
    ref = oracle.move_substances(rho.astype(np.float64), u, v, w, h, dt, split="xz-CellFaceAligned", method=interp)
    assert rel_linf(q, ref) < TOL
    assert st[0]["tables"] == 1 and st[0]["box"] > 0
    assert (st[0]["memory"] > 0) == outside


# grids narrower than the stencil and than a brick, of white noise at large displacements, by tables
# (which the launcher takes from 128 bricks on) and by stencils.  At CFL 7 some corner colours lie within
# FP32 rounding of a cut, which the oracle's FP64 and FP32 cutters settle differently (by 3e-3 of the
# largest value), so every cell must agree with one of the two.
@pytest.mark.parametrize("interp", ["WENO6", "WENO6-optimized"])
@pytest.mark.parametrize("shape,seed,cfl", [((4, 3, 5), 3, 1.5), ((2, 7, 3), 5, 2.0), ((6, 6, 1), 7, 1.0), ((1, 5, 6), 9, 1.0),
                                            ((3, 3, 3), 4, 3.0), ((12, 20, 9), 3, 1.5), ((5, 17, 33), 6, 7.0)])
def test_tables_on_small_grids(forms, oracle, shape, seed, cfl, interp):
    h = 1.0 / 16
    rho, u, v, w, dt = white_noise_scene(*shape, seed, cfl, h)
    refs = [oracle.move_substances(rho.astype(np.float64), u, v, w, h, dt, split="xz-CellFaceAligned", method=interp,
                                   cprec=cp) for cp in (0, 1)]
    for tables in (ALWAYS, NONE):
        q, st = forms.move_substances(rho, u, v, w, h, dt, interp=interp, tables=tables)
        assert np.isfinite(q).all() and rel_linf_either(q, refs) < TOL
        assert st[0]["tables"] == (tables == ALWAYS)


@pytest.mark.parametrize("split", ["none", "xz-CellFaceAligned", "xz-AxisAligned", "x-AxisAligned_z-CellFaceAligned"])
@pytest.mark.parametrize("comp", [-1, 0, 1, 2])
def test_tables_agree_with_stencils(forms, scenes, comp, split):
    # one pass by tables and by stencils: the same points and weights, an interpolated value's FP32
    # rounding apart; bar: half of the pass's own against the oracle
    shape, h = (21, 18, 19), 1.0 / 32
    rho, u, v, w, dt = _box_scene(scenes, shape, 5, 2.0, h)
    q = rho if comp < 0 else (u, v, w)[comp]
    for interp in ("WENO6", "WENO6-optimized"):
        a, st = forms.flux_pass(q, u, v, w, h, dt, split, interp, "WENO6", False, True, comp, ALWAYS)
        b, _ = forms.flux_pass(q, u, v, w, h, dt, split, interp, "WENO6", False, True, comp, NONE)
        assert st[0]["tables"] == 1
        assert np.isfinite(a).all() and rel_linf(a, b) < 0.5 * TOL


@pytest.mark.parametrize("tables", [RULE, ALWAYS])
def test_velocity_step_by_forms(forms, oracle, scenes, tables):
    shape, h = (12, 20, 9), 1.0 / 16
    _, u, v, w, dt = _box_scene(scenes, shape, 11, 2.0, h)
    refs = [oracle.advect_velocity(u, v, w, h, dt, method="WENO6", cprec=cp) for cp in (0, 1)]
    for comp in range(3):
        got, st = forms.advect_velocity(u, v, w, comp, h, dt, tables=tables)
        assert np.isfinite(got).all()
        assert rel_linf_either(got, [r[comp] for r in refs]) < TOL
        assert st[0]["tables"] == tables


@pytest.mark.parametrize("split", ["xz-CellFaceAligned", "xz-AxisAligned", "x-CellFaceAligned_z-AxisAligned"])
@pytest.mark.parametrize("shape", [(1, 5, 4), (19, 6, 33), (14, 9, 8)])
def test_zero_velocity_march_in_any_chunks(forms, oracle, shape, split):
    # chunks of one plane, of some with a remainder, and of all: the same bits, and the oracle's values
    h = 1.0 / 32
    rng = np.random.default_rng(23)
    u, v, w = [np.zeros([s + (a == b) for b, s in enumerate(shape)], dtype=np.float32) for a in range(3)]
    q = np.cumsum(rng.normal(size=shape), axis=2).astype(np.float32)
    ref = oracle.advect_pass(q.astype(np.float64), u, v, w, h, 0.01, split=split, method="WENO6", psi_mode="const",
                             zero_velocity=True, use_integral=False, num_gauss=1)
    whole, _ = forms.flux_pass(q, u, v, w, h, 0.01, split, "WENO6", "const", True, False, zero_chunk=shape[0])
    assert rel_linf(whole, ref) < TOL
    for chunk in (0, 1, 3, 4, 7):
        got, _ = forms.flux_pass(q, u, v, w, h, 0.01, split, "WENO6", "const", True, False, zero_chunk=chunk)
        assert np.array_equal(got, whole)


@pytest.mark.parametrize("method,psi,integral", [("linear", "linear", True), ("WENO6", "WENO6", True), ("WENO6-optimized", "const", False),
                                                 ("1Dy_linear", "const", True), ("1Dy_WENO6", "WENO6", True), ("linear", "const", False)])
def test_zero_velocity_rules(forms, oracle, method, psi, integral):
    shape, h, split = (7, 6, 9), 1.0 / 32, "x-AxisAligned_z-CellFaceAligned"
    rng = np.random.default_rng(29)
    u, v, w = [np.zeros([s + (a == b) for b, s in enumerate(shape)], dtype=np.float32) for a in range(3)]
    q = np.cumsum(rng.normal(size=shape), axis=2).astype(np.float32)
    ref = oracle.advect_pass(q.astype(np.float64), u, v, w, h, 0.01, split=split, method=method, psi_mode=psi,
                             zero_velocity=True, use_integral=integral, num_gauss=1)
    got, _ = forms.flux_pass(q, u, v, w, h, 0.01, split, method, psi, True, integral)
    assert rel_linf(got, ref) < TOL


# the scenes of tests/test_gpu_twisted.py: every face and orientation within its 32 fixed records, and
# some with more, whose pass counts first
@pytest.mark.parametrize("shape,cfl,seed,more", [((12, 14, 13), 6.0, 3, 0), ((32, 8, 32), 40.0, 7, 1)])
def test_twisted_faces_take_their_form(forms, oracle, scenes, shape, cfl, seed, more):
    h = 1.0 / 64
    rho, u, v, w, dt = _box_scene(scenes, shape, seed, cfl, h)
    q, st = forms.move_substances(rho, u, v, w, h, dt)
    ref = oracle.move_substances(rho.astype(np.float64), u, v, w, h, dt, split="xz-CellFaceAligned")
    assert rel_linf(q, ref) < TOL
    assert st[0]["twisted"] > 0 and st[0]["gen_over"] == more
    assert (st[0]["gen_max"] > 32) == bool(more)


def test_subdivided_pieces_by_forms(forms, oracle, scenes):
    shape, h = (8, 7, 9), 1.0 / 64
    rho, u, v, w, dt = _box_scene(scenes, shape, 5, 1.0, h)
    q, _ = forms.move_substances(rho, u, v, w, h, dt, min_area=0.3)
    ref = oracle.move_substances(rho.astype(np.float64), u, v, w, h, dt, split="xz-CellFaceAligned", min_area=0.3)
    assert rel_linf(q, ref) < TOL
