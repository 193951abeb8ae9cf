"""The WENO6 vertex displacements (csrc/fia_kernels.hip vertex_weno_kernel) against the oracle: lattices
of exactly one tile of 16 x 16 (y, z), one vertex more and one less, fields thinner than a stencil,
and an x extent of several chunks, on the cell lattice (two passes a component) and on those of
the face components (one and three passes).  Bar: the FP32 interpolation's, 2e-5 of the largest
displacement.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2e-5


@pytest.mark.parametrize("dim", [-1, 0, 1, 2])
@pytest.mark.parametrize("shape", [(9, 15, 15), (8, 16, 14), (4, 14, 16), (1, 2, 3), (67, 33, 18), (300, 7, 40)])
def test_weno_displacements_match_oracle(fia, oracle, ctx, shape, dim):
    print("case vertices", shape, dim, flush=True)
    h = 0.25
    rng = np.random.default_rng(17)
    fields = [np.cumsum(rng.normal(size=[s + (a == b) for b, s in enumerate(shape)]), axis=(a + 1) % 3).astype(np.float32)
              for a in range(3)]
    top = max(np.abs(f).max() for f in fields)
    dt = h * 2.0 / top
    grid = fia.Grid3D(*shape, h, None, *fields)
    got = fia.backtrace_vertices(ctx, grid, dt, "WENO6", dim).astype(np.float64)
    e = np.array([a == dim for a in range(3)], dtype=np.float64)
    lat = np.stack(np.meshgrid(*[np.arange(s + (a == dim) + 1) for a, s in enumerate(shape)], indexing="ij"), axis=-1)
    ref = oracle.backtrace_vertices(*[f.astype(np.float64) for f in fields], h, dt, "WENO6", comp=dim) / h
    pos = lat - 0.5 * e + got
    assert np.abs(pos - ref).max() < TOL * 2.0
