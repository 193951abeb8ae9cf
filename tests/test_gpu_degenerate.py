"""Degenerate faces (csrc/fia_kernels.hip degenerate_kernel), which eight, four, two or one lane cuts
depending on the length of their list: velocity steps whose component passes list 2 to 6 thousand
faces, 14.8 thousand, 32 thousand and 65 thousand (the pinned walls' corner colours are integers),
against the oracle.  A face there may be settled as the oracle's FP64 or its FP32 cutter does; bar:
the step's, 1e-5 of the component's largest value.
"""
import numpy as np
import pytest

from test_gpu_nonrect import _box_scene

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("shape", [(75, 40, 50), (90, 12, 90), (128, 20, 128)])
def test_degenerate_lists_match_oracle(fia, oracle, ctx, scenes, shape):
    print("case degenerate lists", shape, flush=True)
    h = 1.0 / 32
    _, u, v, w, dt = _box_scene(scenes, shape, 1, 1.0, h)
    grid = fia.Grid3D(*shape, h, None, u.copy(), v.copy(), w.copy())
    fia.advect_velocity_flux_advection_3d(ctx, grid, -1, dt, interpolation_method="linear")
    refs = [oracle.advect_velocity(u, v, w, h, dt, method="linear", cprec=cp) for cp in (0, 1)]
    for a, got in enumerate((grid.u, grid.v, grid.w)):
        err = np.min([np.abs(np.asarray(got, dtype=np.float64) - r[a]) for r in refs], axis=0).max()
        assert err / np.abs(refs[0][a]).max() < TOL, a
