"""Where the multigrid V-cycle's one-block tail begins (csrc/fia_pcg.hip mg_tail_level: its smoothed levels
hold at most 2,048 cells together): a level of exactly that many and one just over, two smoothed levels
in the tail (flat boxes, whose levels shrink slowly), and boxes with one or none, against the Jacobi
solve of the same system.  Bars: those of test_gpu_multigrid_tail.py, both solves to 1e-9 and the
projected velocities within 1e-6 of the largest.  The cycle does not depend on where the tail begins,
so the iterations are those of every level run as a launch of its own (to one, for rounding).
"""
import pytest

from test_gpu_multigrid_tail import _solve, _start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,count", [((32, 64, 64), 28), ((32, 64, 66), 28), ((1, 60, 100), 22), ((1, 2, 2000), 61),
                                         ((25, 77, 64), 28), ((12, 12, 12), 22)])
def test_tail_cutoff_solves_as_jacobi(fia, shape, count):
    print("case tail cut-off", shape, flush=True)
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
    assert abs(it - count) <= 1
    for x, y in ((a.u, b.u), (a.v, b.v), (a.w, b.w)):
        assert float((x - y).abs().max()) <= 1e-6 * max(1.0, float(y.abs().max()))
