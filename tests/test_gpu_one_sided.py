"""The terrain solve with smoothing on one side of the coarse correction only, or
on neither, against the oracle's full cycle.

These cycles too leave out what changes no iterate, and keep the finest levels
colour-split: without post-smoothing both colours are corrected and the CG's
sums are a pass of their own, without pre-smoothing the right-hand side itself is
restricted. The same bounds as for smoothing on both sides: 1e-10 of the largest
value after a few iterations whose sums have up to n terms (a colour left
uncorrected, or a residual of the wrong cells, shows at 1e-3). Sizes: pairs and
rows past and short of the blocks, several chunks of levels, one level, and a
second level that takes its coefficients from the metrics.
"""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu


def _solve(hip, orc, n, nu, its):
    from aeolus_hip.terrain import AnelasticTerrainSimulation, TerrainFollowingGrid, gaussian_hills
    dx, lid = 100.0, 3200.0
    phys = dict(rho0=1.2, Hs=8000.0, theta0=300.0, gamma=0.003, g_accel=9.81)
    ext = (n[0] * dx, n[1] * dx, lid)
    h = gaussian_hills(n, (dx, dx), n=3, seed=5, height=(100.0, 400.0), half_width=(300.0, 800.0))
    tg = TerrainFollowingGrid(hip.Grid(n, ext, halo=3), h, lid)
    sim = AnelasticTerrainSimulation(tg, tol=1e-30, maxit=its, nu1=nu[0], nu2=nu[1], **phys)
    core = orc.TerrainCore(orc.Grid(n, ext, halo=3), tg.plane, lid, scheme="weno_z5", **phys).use_multigrid(*nu)
    b = np.random.default_rng(sum(n)).standard_normal(n)
    x, it, _ = core.solve(b, tol=1e-30, maxit=its)
    got = sim.solve(hip.DeviceArray.from_numpy(np.asfortranarray(b))).download()
    assert it == its and sim.solver_stats()["iterations"] == its
    return got, x


@pytest.mark.parametrize("nu", [(1, 0), (3, 0), (0, 1), (0, 2), (0, 0)])
@pytest.mark.parametrize("n", [(8, 8, 8), (9, 7, 6), (72, 24, 16), (136, 40, 24), (16, 264, 48)])
def test_cycle(hip, orc, n, nu):
    got, x = _solve(hip, orc, n, nu, 3)
    assert rel_err(got, x) < 1e-10


@pytest.mark.parametrize("nu", [(2, 0), (0, 2)])
def test_second_level_from_the_metrics(hip, orc, nu):
    n = (584, 640, 36)
    assert n[0] * n[1] * n[2] // 8 >= 3 << 19
    got, x = _solve(hip, orc, n, nu, 1)
    assert rel_err(got, x) < 1e-10
