"""The table quadrature (csrc/fia_kernels.hip piece_brick_kernel), which serves grids of at least 128
bricks of 4 x 8 x 16 cells, against the FP64 oracle: grids of whole bricks and with a remainder on
every axis, boxes thinner than a brick (clamped stencils in the staged box), flows that keep a
brick's pieces inside the staged box and flows whose shear throws some out of it (the last three
shapes), both interpolations, and the staggered grids of the velocity step.  The bar is the
density step's.
"""
import numpy as np
import pytest

from conftest import rel_linf
from test_gpu_nonrect import _box_scene

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("interp", ["WENO6", "WENO6-optimized"])
@pytest.mark.parametrize("shape,cfl", [((16, 32, 128), 1.0), ((17, 33, 81), 2.0), ((66, 9, 50), 3.0), ((5, 71, 131), 4.0), ((36, 40, 40), 4.0)])
def test_density_step_on_bricks_matches_oracle(fia, oracle, ctx, scenes, shape, cfl, interp):
    print("case bricks", shape, cfl, interp, flush=True)
    h = 1.0 / 64
    rho, u, v, w, dt = _box_scene(scenes, shape, 11, cfl, h)
    grid = fia.Grid3D(*shape, h, rho.copy(), u, v, w)
    fia.move_substances_3d(ctx, grid, 0, dt, split_method="xz-CellFaceAligned", interpolation_method=interp)
    ref = oracle.move_substances(rho.astype(np.float64), u, v, w, h, dt, split="xz-CellFaceAligned", method=interp)
    assert rel_linf(grid.density, ref) < TOL


def test_velocity_step_on_bricks_matches_oracle(fia, oracle, ctx, scenes):
    shape, h = (30, 33, 50), 1.0 / 64
    print("case velocity bricks", shape, flush=True)
    _, u, v, w, dt = _box_scene(scenes, shape, 13, 2.0, h)
    grid = fia.Grid3D(*shape, h, None, u.copy(), v.copy(), w.copy())
    fia.advect_velocity_flux_advection_3d(ctx, grid, -1, dt, interpolation_method="WENO6")
    # corners of pinned vertices on cut lines: the FP32 or the FP64 cutter's pieces, cell by cell
    refs = [oracle.advect_velocity(u, v, w, h, dt, method="WENO6", cprec=cp) for cp in (0, 1)]
    for a, got in enumerate((grid.u, grid.v, grid.w)):
        err = np.min([np.abs(np.asarray(got, dtype=np.float64) - r[a]) for r in refs], axis=0).max()
        assert err / np.abs(refs[0][a]).max() < TOL, a
