"""The terrain operator L φ = B(Gφ) in one pass, against the oracle's two.

The kernel carries ρ, ρJ and 1/ρJ up a chunk by their ratio between levels:
over at most 64 levels each is within 64 x 2 roundings (1.4e-14) of the value
the oracle evaluates (on these small grids the chunks have 1 to 7 levels; 43 and
64 in test_gpu_long_chunks.py), and the terms of L φ are at most about ten times its
largest value (steep hills, dz << dx), so 1e-12 holds; a coefficient of the
wrong level or column is off by dz/Hs = 1e-3 or more. Sizes: columns and rows
one past, one short of and well below the block's 64 x 4; chunks of one level
and of several with a remainder.
"""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(6, 6, 8), (63, 5, 13), (65, 9, 67), (130, 7, 50), (64, 72, 131), (8, 300, 66)])
def test_apply(hip, orc, n):
    from aeolus_hip.terrain import AnelasticTerrainSimulation, TerrainFollowingGrid, gaussian_hills
    dx, lid = 100.0, 3200.0
    phys = dict(rho0=1.2, Hs=8000.0, theta0=300.0, gamma=0.003, g_accel=9.81)
    ext = (n[0] * dx, n[1] * dx, lid)
    h = gaussian_hills(n, (dx, dx), n=3, seed=5, height=(100.0, 400.0), half_width=(300.0, 800.0))
    tg = TerrainFollowingGrid(hip.Grid(n, ext, halo=3), h, lid)
    sim = AnelasticTerrainSimulation(tg, **phys)
    core = orc.TerrainCore(orc.Grid(n, ext, halo=3), tg.plane, lid, scheme="weno_z5", **phys)
    x = np.asfortranarray(np.random.default_rng(sum(n)).standard_normal(n))
    got = sim.apply(hip.DeviceArray.from_numpy(x)).download()
    assert rel_err(got, core.apply(x)) < 1e-12
