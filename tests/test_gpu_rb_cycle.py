"""The red-black V-cycle without its redundant work (the colour whose residual
vanishes, the correction the next pass overwrites, the mean removals inside
the cycle, the clearing of phi), against the oracle's full cycle.

The two are the same in exact arithmetic, so the CG's iterates after a fixed
number of iterations agree to rounding: three iterations of a cycle whose
sums have up to n terms, within 1e-10 of the largest value (a residual
formed on the wrong cells, or a missing correction, shows at 1e-3). Sizes:
pairs and rows past and short of the blocks, chunks of 2 and 4 levels (32 in
test_gpu_long_chunks.py), mirror boundaries on every axis.
"""
import ctypes

import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu

ITS = 3


@pytest.mark.parametrize("nu", [(2, 2), (1, 1), (2, 0)])
@pytest.mark.parametrize("n", [(8, 8, 8), (72, 24, 16), (136, 40, 24), (16, 264, 48), (48, 48, 96)])
def test_terrain_cycle(hip, orc, n, nu):
    from aeolus_hip.terrain import AnelasticTerrainSimulation, TerrainFollowingGrid, gaussian_hills
    dx, lid = 100.0, 3200.0
    phys = dict(rho0=1.2, Hs=8000.0, theta0=300.0, gamma=0.003, g_accel=9.81)
    ext = (n[0] * dx, n[1] * dx, lid)
    h = gaussian_hills(n, (dx, dx), n=3, seed=5, height=(100.0, 400.0), half_width=(300.0, 800.0))
    tg = TerrainFollowingGrid(hip.Grid(n, ext, halo=3), h, lid)
    sim = AnelasticTerrainSimulation(tg, tol=1e-30, maxit=ITS, nu1=nu[0], nu2=nu[1], **phys)
    core = orc.TerrainCore(orc.Grid(n, ext, halo=3), tg.plane, lid, scheme="weno_z5", **phys).use_multigrid(*nu)
    b = np.random.default_rng(sum(n)).standard_normal(n)
    x, it, _ = core.solve(b, tol=1e-30, maxit=ITS)
    got = sim.solve(hip.DeviceArray.from_numpy(np.asfortranarray(b))).download()
    assert it == ITS and sim.solver_stats()["iterations"] == ITS
    assert rel_err(got, x) < 1e-10


@pytest.mark.parametrize("vcycle,its,tol", [("f64", ITS, 1e-10), ("f32", 1, 2e-5)])
@pytest.mark.parametrize("bcs", [("periodic", "periodic", "neumann"), ("neumann", "periodic", "periodic"), ("neumann",) * 3])
@pytest.mark.parametrize("n", [(8, 16, 8), (40, 24, 16), (136, 8, 32)])
def test_uniform_cycle(hip, orc, n, bcs, vcycle, its, tol):
    # FP32 levels: one iteration (the FP32 cycle's CG takes the flexible β, another
    # number where the cycle is not symmetric): 2 x 8 half-sweeps and two
    # transfers per level pair, each within about 10 FP32 roundings of 6e-8
    L = orc.lib()
    h = L.orc_mg_create(*n, 1.0, 1.3, 0.7, *[orc.BCS[q] for q in bcs], None, None, None, None, 2, 2, 4, 0, 1.0)
    b = np.asfortranarray(np.random.default_rng(sum(n)).standard_normal(n))
    x = np.zeros(n, order="F")
    it, res, bn = ctypes.c_int(), ctypes.c_double(), ctypes.c_double()
    L.orc_mgpcg_solve(h, orc.ptr(x), orc.ptr(b), 1e-30, its, ctypes.byref(it), ctypes.byref(res), ctypes.byref(bn))
    L.orc_mg_destroy(h)
    s = hip.MGPreconditionedCG(n, (1.0, 1.3, 0.7), bcs=bcs, tol=1e-30, maxit=its, vcycle=vcycle)
    got = hip.solve_interior(s, b)
    assert hip.solver_stats(s)[0] == it.value == its
    assert rel_err(got, x) < tol
