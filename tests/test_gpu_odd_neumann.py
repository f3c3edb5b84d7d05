"""The column solver with a Neumann y-axis of odd length, against the oracle.

The cosine transform reorders an axis by its even places up and its odd ones
down: an odd length has one even place more. Lengths of one factor and of
several, the smallest, and several blocks of columns; the x-axis periodic and
Neumann. A few hundred roundings of a direct solve, against the largest value:
1e-12, as for even lengths; a place taken twice or from the next plane shows at
1e-2.
"""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bcx", ["periodic", "neumann"])
@pytest.mark.parametrize("size", [(8, 3, 4), (16, 9, 7), (48, 5, 12), (60, 45, 6), (64, 15, 33), (250, 125, 3)])
def test_column_solver(hip, orc, size, bcx):
    extent = (100.0, 60.0, 80.0)
    zf = np.concatenate([[0.0], np.cumsum(np.linspace(1.0, 2.0, size[2]))])
    zf *= extent[2] / zf[-1]
    g, og = (G(size, extent, halo=1, zf=zf) for G in (hip.Grid, orc.Grid))
    src = np.asfortranarray(np.random.default_rng(size[0]).normal(size=size))
    ref = orc.stretched_column_solver(og, bcx, "neumann").solve(src)
    dzc, dzf = g.interior_dz()
    s = hip.ColumnTridiagonalSolver.stretched(size, (g.dx, g.dy), dzc, dzf, bc_x=bcx, bc_y="neumann")
    got = hip.solve_interior(s, src)
    assert rel_err(got, ref) <= 1e-12
    assert np.array_equal(hip.solve_interior(s, src), got)  # nothing left in the spectrum's next plane
