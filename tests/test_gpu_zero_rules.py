"""The zero-velocity pass by the kernels that are compiled for one interpolation's quadrature
(csrc/fia_kernels.hip zero_velocity_face_kernel), against the oracle: integral and not, with both axes
of a face cut, one, and none.  Bar: the pass's, 1e-5 of the field's largest value.
"""
import numpy as np
import pytest

from conftest import rel_linf

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("split", ["xz-CellFaceAligned", "x-AxisAligned_z-CellFaceAligned", "none"])
@pytest.mark.parametrize("method,psi,integral", [("linear", "linear", True), ("WENO6", "WENO6", True), ("WENO6", "const", False),
                                                 ("WENO6-optimized", "WENO6", True), ("WENO6-optimized", "const", False),
                                                 ("1Dy_linear", "const", True), ("1Dy_WENO6", "WENO6", True),
                                                 ("1Dy_WENO6", "const", False)])
@pytest.mark.parametrize("shape", [(1, 5, 4), (19, 6, 33)])
def test_zero_velocity_rule_matches_oracle(fia, oracle, ctx, shape, method, psi, integral, split):
    print("case zero rule", shape, method, psi, integral, split, flush=True)
    h = 1.0 / 32
    rng = np.random.default_rng(29)
    u, v, w = [np.zeros([s + (a == b) for b, s in enumerate(shape)], dtype=np.float32) for a in range(3)]
    q = np.cumsum(rng.normal(size=shape), axis=2).astype(np.float32)
    ref = oracle.advect_pass(q.astype(np.float64), u, v, w, h, 0.01, split=split, method=method, psi_mode=psi,
                             zero_velocity=True, use_integral=integral, num_gauss=1)
    grid = fia.Grid3D(*shape, h, None, u, v, w)
    got = q.copy()
    fia.advect_flux_pass(ctx, grid, got, 0.01, split, method, psi, True, integral, 1)
    assert rel_linf(got, ref) < TOL
