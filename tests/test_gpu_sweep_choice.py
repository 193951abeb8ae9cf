"""The default form of the Jacobi iteration (csrc/fia_pcg.hip pcg_fused_pays, fused_plan): one sweep,
in chunks that put one, two or three blocks on every CU, and two sweeps on thin boxes.  A solve's bits
follow its form and its chunks (the order of the partial sums), so the default must give exactly the
bits of the form and chunk that the rule's costs name, and not those of the other form or of another
chunk.  Costs in us, one sweep with 1, 2, 3 blocks per CU and two sweeps (256 CUs, 3 resident blocks each):
64^3 12.5 16.3 17.6, 16.3; 128^3 28.2 24.8 26.2, 35.2; 96x128x128 23.7 22.0 21.9, 28.8; 300x300x3
64.2 47.6 47.7, 31.7; 256x256x16 46.2 36.2 39.1, 33.5; 97x194x22 23.7 22.0 21.9, 19.7; 4000x4x4 46.2 36.2
39.1, 25.7.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(fia, c, shape, start, **tuning):
    import torch
    nx, ny, nz = shape
    c.set_tuning(shape, **tuning)
    u, v, w = [torch.tensor(f, device="cuda:0") for f in start]
    grid = fia.Grid3D(nx, ny, nz, 1.0 / max(shape), None, u, v, w)
    grid.density = None
    torch.cuda.synchronize()
    it, res = fia.calc_pressure_gradient_term_3d(c, grid, rel_tol=1e-6)
    return it, grid.pressure.cpu().numpy()


@pytest.mark.parametrize("shape,fused,chunk,other", [((64, 64, 64), 1, 1, 2), ((128, 128, 128), 1, 4, 3), ((96, 128, 128), 1, 2, 3),
                                                     ((300, 300, 3), 0, 8, 12), ((256, 256, 16), 0, 6, 8), ((97, 194, 22), 0, 2, 3),
                                                     ((4000, 4, 4), 0, 6, 8)])
def test_default_form_and_chunk(fia, shape, fused, chunk, other):
    print("case sweep choice", shape, flush=True)
    nx, ny, nz = shape
    rng = np.random.default_rng(3)
    start = [rng.normal(size=s).astype(np.float32) for s in ((nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1))]
    c = fia.Context(0)
    try:
        c.set_pressure_preconditioner("jacobi")
        it, p = _solve(fia, c, shape, start)
        same_it, same = _solve(fia, c, shape, start, pcg_fused=fused, pcg_chunk_x=chunk)
        _, rechunked = _solve(fia, c, shape, start, pcg_fused=fused, pcg_chunk_x=other)
        _, reformed = _solve(fia, c, shape, start, pcg_fused=1 - fused)
    finally:
        c.close()
    assert it == same_it and np.array_equal(p, same)
    assert not np.array_equal(p, rechunked) and not np.array_equal(p, reformed)
