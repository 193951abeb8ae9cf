"""The multigrid V-cycle's one-block tail (csrc/fia_pcg.hip mg_tail_body) and the pinned cell.

Grids whose coarse levels give the tail nothing but the coarsest level, one smoothed level, several,
odd edges and edges of one cell, and coarsest levels of one cell to 256, against the Jacobi solve of
the same system: both to 1e-9, so their projected velocities agree to 1e-6 of the largest (a factor
of 1000 over the tolerance).  The cycle is a fixed symmetric operator, so CG's count stays that of
multigrid: under 60 where Jacobi takes hundreds.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _start(shape, seed):
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    f = [rng.normal(size=s).astype(np.float32) for s in ((nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1))]
    for a in range(3):
        for end in (0, -1):
            f[a][tuple(slice(None) if b != a else end for b in range(3))] = 0
    return f


def _solve(fia, c, start, solid, tol):
    import torch
    nx, ny, nz = start[0].shape[0] - 1, start[0].shape[1], start[0].shape[2]
    u, v, w = [torch.tensor(f, device="cuda:0") for f in start]
    grid = fia.Grid3D(nx, ny, nz, 1.0 / max(nx, ny, nz), None, u, v, w)
    grid.density = None
    torch.cuda.synchronize()
    it, res = fia.calc_pressure_gradient_term_3d(c, grid, solid=solid, rel_tol=tol)
    return grid, it, res


@pytest.mark.parametrize("shape", [(8, 8, 8), (12, 14, 13), (33, 34, 35), (40, 9, 17), (1, 40, 33), (2, 3, 300),
                                   (50, 77, 64), (96, 96, 96)])
def test_tail_solves_as_jacobi(fia, shape):
    print("case tail", shape, flush=True)
    start = _start(shape, 5)
    c = fia.Context(0)
    try:
        a, it, res = _solve(fia, c, start, None, 1e-9)
        c.set_pressure_preconditioner("jacobi")
        b, itj, resj = _solve(fia, c, start, None, 1e-9)
    finally:
        c.close()
    print("iterations %d, jacobi %d" % (it, itj), flush=True)
    assert res <= 1e-9 and resj <= 1e-9
    assert it <= 60
    for x, y in ((a.u, b.u), (a.v, b.v), (a.w, b.w)):
        assert float((x - y).abs().max()) <= 1e-6 * max(1.0, float(y.abs().max()))


@pytest.mark.parametrize("tail", [0, 1, 15, 16, 16384, 16385, 20000, 32 ** 3 - 2])
def test_last_fluid_cell_is_pinned(fia, ctx, tail):
    import torch
    print("case pinned cell", tail, flush=True)
    n = 32
    solid = torch.zeros(n ** 3, dtype=torch.uint8, device="cuda:0")
    solid[n ** 3 - tail:] = 1
    if tail > 16:
        solid[n ** 3 - 1 - tail // 2] = 0   # a lone fluid cell inside the solid tail
    pin = int(torch.nonzero(solid == 0)[-1])
    grid, it, res = _solve(fia, ctx, _start((n, n, n), 6), solid.view(n, n, n), 1e-6)
    p = grid.pressure.reshape(-1)
    assert float(p[pin]) == 0.0
    if pin == n ** 3 - 1 - tail:   # a cell of the fluid's body: its neighbours are not 0 by accident
        assert float(p[pin - 1].abs() + p[pin - n].abs()) > 0.0
    assert res <= 1e-6


def test_all_solid_is_refused(fia, ctx):
    import torch
    with pytest.raises(fia.FiaError) as e:
        _solve(fia, ctx, _start((9, 9, 9), 7), torch.ones((9, 9, 9), dtype=torch.uint8, device="cuda:0"), 1e-6)
    assert e.value.status == 1
