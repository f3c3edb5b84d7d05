"""The marching kernels at the chunk lengths of large grids, against the oracle.

The levels a block marches follow the number of blocks, so small grids run short
chunks. Grids of a few columns by thousands of rows have as many blocks as the
large ones at a thousandth of their cells, and march the longest chunks, 16
levels (8 in the scalar kernel), 32, 43 and 64, with a shorter last one. Each test
first asserts the length it is about (aeo_launch_levels). Tolerances are those
of the small grids: a value carried up 64 levels by its ratio is within 64 x 2
roundings, 1.4e-14, of the one the oracle evaluates; a window that is not
rotated, or a flux carried past its level, shows at 1e-2 or more.
"""
import ctypes

import numpy as np
import pytest

from helpers import rand_storage, rel_err

pytestmark = pytest.mark.gpu

PHYS = dict(rho0=1.2, Hs=8000.0, theta0=300.0, gamma=0.003, g_accel=9.81)


def _levels(kernel, n):
    from aeolus_hip import _lib
    k = ctypes.c_int()
    _lib.check(_lib.load().aeo_launch_levels(kernel.encode(), *n, ctypes.byref(k)))
    return k.value


def _fields(orc, og, seeds):
    out = [rand_storage(og.storage, s) for s in seeds]
    for a, loc in zip(out, (1, 2, 3, 0)):
        orc.fill_halos(og, a, loc, ("periodic",) * 3)
    return out


@pytest.mark.parametrize("scheme,H", [("weno_z5", 3), ("weno_z7", 4), ("centered", 2)])
def test_advection(hip, orc, scheme, H):
    n = (6, 2043, 31)
    assert (_levels("tendency", n), _levels("scalar", n), _levels("limited", n)) == (16, 8, 16)
    g, og = (G(n, (3.0, 1.0, 2.0), halo=H) for G in (hip.Grid, orc.Grid))
    u, v, w, phi = _fields(orc, og, range(7, 11))
    dev = [hip.DeviceArray.from_numpy(a) for a in (u, v, w, phi)]
    I = og.interior
    ref = orc.advect_momentum(og, og.zeros(), og.zeros(), og.zeros(), u, v, w, scheme)
    out = [g.field() for _ in range(3)]
    hip.advection_scheme(scheme, g).momentum(*out, *dev[:3])
    for a, b in zip(out, ref):
        assert rel_err(a.download()[I], b[I]) <= 1e-12
    t = g.field()
    hip.advection_scheme(scheme, g)(t, *dev)
    assert rel_err(t.download()[I], orc.advect_scalar(og, og.zeros(), u, v, w, phi, scheme)[I]) <= 1e-12
    phi = np.abs(phi)
    t = g.field()
    hip.advect_positive(g, t, *dev[:3], hip.DeviceArray.from_numpy(phi), 0.001, scheme=scheme, accumulate=False)
    ref = orc.advect_positive(og, og.zeros(), u, v, w, phi, 0.001, scheme=scheme, accumulate=False)
    assert rel_err(t.download()[I], ref[I]) <= 1e-12


def test_step(hip, orc):
    """The step's tendencies (four fields, 16-level chunks) with a stretched column
    (the spectral solver takes no thousands of rows)."""
    from aeolus_hip import workloads as W
    n = (480, 250, 31)
    assert _levels("tendency", n) == 16
    zf, Lz = W.dcbl_faces(n[2])
    ext = (20.0 * n[0], 20.0 * n[1], Lz)
    g, og = hip.Grid(n, ext, halo=3, zf=zf), orc.Grid(n, ext, halo=3, zf=zf)
    state = W.dcbl_state(g)
    rng = np.random.default_rng(7)
    for a in state[:2]:
        a[g.interior] += 0.5 * rng.uniform(-1, 1, size=a[g.interior].shape)
    sim = hip.BoussinesqSimulation(g, scheme="weno_z5", **W.DCBL_PHYS)
    sim.set(*state)
    sim.step(0.5)
    got = sim.state()
    ost = orc.Stepper(og, scheme="weno_z5", **W.DCBL_PHYS)
    ref = [np.asfortranarray(a.copy()) for a in state]
    p = og.zeros()
    ost.euler(*ref, p, 0.5)
    for name, r in zip(("u", "v", "w", "theta"), ref):
        assert rel_err(got[name], r) <= 1e-12, name


def _terrain(hip, orc, n, **kw):
    from aeolus_hip.terrain import AnelasticTerrainSimulation, TerrainFollowingGrid, gaussian_hills
    dx, lid = 100.0, 3200.0
    ext = (n[0] * dx, n[1] * dx, lid)
    h = gaussian_hills(n, (dx, dx), n=40, seed=5, height=(100.0, 400.0), half_width=(300.0, 800.0))
    tg = TerrainFollowingGrid(hip.Grid(n, ext, halo=3), h, lid)
    og = orc.Grid(n, ext, halo=3)
    return AnelasticTerrainSimulation(tg, **PHYS, **kw), orc.TerrainCore(og, tg.plane, lid, scheme="weno_z5", **PHYS), tg, og


@pytest.mark.parametrize("n,kc", [((6, 3070, 86), 43), ((6, 3070, 127), 64)])
def test_terrain_apply(hip, orc, n, kc):
    assert _levels("terrain_apply", n) == kc
    sim, core, _, _ = _terrain(hip, orc, n)
    x = np.asfortranarray(np.random.default_rng(sum(n)).standard_normal(n))
    got = sim.apply(hip.DeviceArray.from_numpy(x)).download()
    assert rel_err(got, core.apply(x)) < 1e-12


@pytest.mark.parametrize("flux,tol", [("f64", 1e-12), ("f32", 1e-4)])
def test_terrain_tendencies(hip, orc, flux, tol):
    from test_gpu_terrain_core import _random_state, _up
    n, lid = (6, 2046, 63), 3200.0
    assert _levels("terrain_tendency", n) == 32
    sim, core, tg, og = _terrain(hip, orc, n, flux_precision=flux)
    u, v, w, th = _random_state(og, core, 20, U=10.0)
    ref = core.tendencies(u, v, w, th)
    I, H = og.interior, og.H
    if flux == "f32":  # its form less θ_c·(B u)/(ρ̄J), added back
        J = (lid - tg.plane[H:H + og.Nx, H:H + og.Ny]) / lid
        ref[3][I] += th[I] * core.divergence(u, v, w) / (core.density(0)[I] * J[:, :, None])
    got = sim.tendencies([_up(a) for a in (u, v, w, th)])
    for a, b, name in zip(got, ref, ("tu", "tv", "tw", "ttheta")):
        err = rel_err(a.download()[I], b[I])
        assert err <= tol, (name, err)


@pytest.mark.parametrize("n,its,levels", [((8, 4096, 62), 3, [(32, 16)]), ((16, 8192, 124), 1, [(32, 16), (32, 16)])])
def test_terrain_cycle(hip, orc, n, its, levels):
    """The red-black V-cycle's finest levels in chunks of 32 levels (transfers:
    16) and a remainder; the second grid's second level takes its coefficients
    from the metrics too."""
    for l, (kc, kp) in enumerate(levels):
        m = tuple(q >> l for q in n)
        assert (_levels("terrain_smooth", m), _levels("terrain_prolong", m)) == (kc, kp) and m[2] % kc
    assert (n[0] * n[1] * n[2] // 8 >= 3 << 19) == (len(levels) == 2)
    sim, core, _, _ = _terrain(hip, orc, n, tol=1e-30, maxit=its, nu1=2, nu2=2)
    core.use_multigrid(2, 2)
    b = np.random.default_rng(sum(n)).standard_normal(n)
    x, it, _ = core.solve(b, tol=1e-30, maxit=its)
    got = sim.solve(hip.DeviceArray.from_numpy(np.asfortranarray(b))).download()
    assert it == its and sim.solver_stats()["iterations"] == its
    assert rel_err(got, x) < 1e-10
