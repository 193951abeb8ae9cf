"""The zero-velocity pass of the WENO6 rule in chunks of x planes (csrc/fia_kernels.hip
zero_velocity_weno_kernel) against the oracle: chunks of one plane, of four with a remainder of one and
three planes, and rows that end inside a block, for each split that cuts
both axes of a face and one that does not.  Bar: the pass's, 1e-5 of the field's largest value.
"""
import numpy as np
import pytest

from conftest import rel_linf

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("split", ["xz-CellFaceAligned", "xz-AxisAligned", "x-CellFaceAligned_z-AxisAligned"])
@pytest.mark.parametrize("shape", [(1, 5, 4), (19, 6, 33), (113, 50, 47), (111, 47, 50)])
def test_zero_velocity_pass_matches_oracle(fia, oracle, ctx, scenes, shape, split):
    print("case zero velocity", shape, split, flush=True)
    h = 1.0 / 32
    rng = np.random.default_rng(23)
    u, v, w = [np.zeros([s + (a == b) for b, s in enumerate(shape)], dtype=np.float32) for a in range(3)]
    q = np.cumsum(rng.normal(size=shape), axis=2).astype(np.float32)
    ref = oracle.advect_pass(q.astype(np.float64), u, v, w, h, 0.01, split=split, method="WENO6", psi_mode="const",
                             zero_velocity=True, use_integral=False, num_gauss=1)
    grid = fia.Grid3D(*shape, h, None, u, v, w)
    got = q.copy()
    fia.advect_flux_pass(ctx, grid, got, 0.01, split, "WENO6", "const", True, False, 1)
    assert rel_linf(got, ref) < TOL
