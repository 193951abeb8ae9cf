"""The fused Jacobi sweep's default chunks (csrc/fia_pcg.hip fused_chunks): grids that take one, two
and three blocks per CU, and one past the cached sizes, against the two-sweep iteration.  Both
solve to 1e-8; CG's iterates agree to rounding, so the counts may differ by a few of hundreds and
the projected velocities by the two solves' own residuals: 1e-6 of the largest velocity leaves a
factor of 100 over the tolerance.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(21, 18, 70), (64, 64, 64), (40, 130, 66), (96, 96, 96), (161, 160, 164)])
def test_default_chunks_reach_the_two_sweep_solution(fia, scenes, shape):
    import torch
    print("case fused chunks", shape, flush=True)
    rng = np.random.default_rng(3)
    nx, ny, nz = shape
    start = [rng.normal(size=s).astype(np.float32) for s in ((nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1))]
    for a, f in enumerate(start):
        f[tuple(slice(None) if b != a else 0 for b in range(3))] = 0
        f[tuple(slice(None) if b != a else -1 for b in range(3))] = 0
    c = fia.Context(0)
    try:
        c.set_pressure_preconditioner("jacobi")
        got = []
        for fused in (-1, 0):
            c.set_tuning(shape, pcg_fused=fused)
            u, v, w = [torch.tensor(f, device="cuda:0") for f in start]
            grid = fia.Grid3D(nx, ny, nz, 1.0 / 64, None, u, v, w)
            grid.density = None
            torch.cuda.synchronize()
            it, res = fia.calc_pressure_gradient_term_3d(c, grid, rel_tol=1e-8)
            assert res <= 1e-8
            got.append((it, grid.u, grid.v, grid.w))
    finally:
        c.close()
    print("iterations %d and %d" % (got[0][0], got[1][0]), flush=True)
    assert abs(got[0][0] - got[1][0]) <= 2 + 0.02 * got[1][0]
    for a, b in zip(got[0][1:], got[1][1:]):
        assert float((a - b).abs().max()) <= 1e-6 * float(b.abs().max())
