"""The terrain grid's second level from the metrics and colour-split (grids
whose second level has at least 3·2^19 cells), against the oracle's cycle with
the stored coefficients.

One iteration of the CG, x = α z with z one V-cycle: its sums have up to n
terms and the carried coefficients are within about 64 ulp of the stored ones,
so 1e-10 of the largest value holds; a coefficient of the wrong face, or a
value read from the wrong colour's half, shows at 1e-3. The levels below the
second are the generic ones; the second level's 16 and 18 levels are two chunks
of 8, and 10 and 8 (32 in test_gpu_long_chunks.py), the widths whole and
partial blocks.
"""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(640, 632, 32), (584, 640, 36)])
def test_one_cycle(hip, orc, n):
    from aeolus_hip.terrain import AnelasticTerrainSimulation, TerrainFollowingGrid, gaussian_hills
    assert n[0] * n[1] * n[2] // 8 >= 3 << 19
    dx, lid = 100.0, 3200.0
    phys = dict(rho0=1.2, Hs=8000.0, theta0=300.0, gamma=0.003, g_accel=9.81)
    ext = (n[0] * dx, n[1] * dx, lid)
    h = gaussian_hills(n, (dx, dx), n=3, seed=5, height=(100.0, 400.0), half_width=(300.0, 800.0))
    tg = TerrainFollowingGrid(hip.Grid(n, ext, halo=3), h, lid)
    sim = AnelasticTerrainSimulation(tg, tol=1e-30, maxit=1, **phys)
    core = orc.TerrainCore(orc.Grid(n, ext, halo=3), tg.plane, lid, scheme="weno_z5", **phys).use_multigrid(2, 2)
    b = np.random.default_rng(sum(n)).standard_normal(n)
    x, it, _ = core.solve(b, tol=1e-30, maxit=1)
    got = sim.solve(hip.DeviceArray.from_numpy(np.asfortranarray(b))).download()
    assert it == 1 and sim.solver_stats()["iterations"] == 1
    assert rel_err(got, x) < 1e-10
