"""Twisted faces (csrc/fia_kernels.hip general_*): the pieces of a face and orientation are stored in
a fixed number of records, or counted first where some pair has more (a flow that stretches faces
over tens of cells) or minimal_area < 1 sends every face there.  Each form against the FP64 oracle,
at the density step's bar.
"""
import numpy as np
import pytest

from conftest import rel_linf
from test_gpu_nonrect import _box_scene

pytestmark = pytest.mark.gpu

TOL = 1e-5


# 16 - 28 pieces a twisted face (fixed records), and up to 124 (counted)
@pytest.mark.parametrize("shape,cfl,seed", [((12, 14, 13), 6.0, 3), ((32, 8, 32), 40.0, 7)])
def test_twisted_faces_match_oracle(fia, oracle, scenes, shape, cfl, seed):
    print("case twisted", shape, cfl, flush=True)
    h = 1.0 / 64
    rho, u, v, w, dt = _box_scene(scenes, shape, seed, cfl, h)
    c = fia.Context(0)
    try:
        c.set_timing(True)
        c.reset_stats()
        grid = fia.Grid3D(*shape, h, rho.copy(), u, v, w)
        fia.move_substances_3d(c, grid, 0, dt, split_method="xz-CellFaceAligned", interpolation_method="WENO6")
        st = c.stats()
    finally:
        c.close()
    print("twisted faces %d, pieces %d" % (st["twisted_faces"], st["general_pieces"]), flush=True)
    assert st["twisted_faces"] > 0
    ref = oracle.move_substances(rho.astype(np.float64), u, v, w, h, dt, split="xz-CellFaceAligned")
    assert rel_linf(grid.density, ref) < TOL


def test_subdivided_pieces_match_oracle(fia, oracle, ctx, scenes):
    shape, h = (8, 7, 9), 1.0 / 64
    print("case minimal area 0.3", shape, flush=True)
    rho, u, v, w, dt = _box_scene(scenes, shape, 5, 1.0, h)
    grid = fia.Grid3D(*shape, h, rho.copy(), u, v, w)
    fia.move_substances_3d(ctx, grid, 0, dt, split_method="xz-CellFaceAligned", interpolation_method="WENO6",
                           minimal_area=0.3)
    ref = oracle.move_substances(rho.astype(np.float64), u, v, w, h, dt, split="xz-CellFaceAligned", min_area=0.3)
    assert rel_linf(grid.density, ref) < TOL
