"""The sound-proof core's Runge-Kutta step, whose combinations ride in the
correction and the shell pass and whose divergence is formed in the row
transform, against the same step composed on the host from its Euler steps.

FP64: the combination's two products and sum round as on the host (the
multiplied values may round once less): 3 stages of 1e-15 on values whose
later tendencies and projection amplify by a few, 1e-13. FP32: 1e-5, three
stages of 6e-8 likewise. The whole storage is compared, halo shell included.
Lateral walls take the form with the divergence pass.
"""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(0, 1e-13), (1, 1e-5)])
@pytest.mark.parametrize("bcs", [("periodic", "periodic", "wall"), ("noflux", "periodic", "wall")])
@pytest.mark.parametrize("n", [(8, 6, 5), (60, 9, 13), (30, 40, 16)])
def test_rk3_is_its_euler_steps(hip, n, bcs, prec, tol):
    from aeolus_hip.anelastic import AnelasticSimulation, isothermal_reference
    g = hip.Grid(n, (n[0] * 100.0, n[1] * 100.0, n[2] * 100.0), halo=2)
    kw = dict(nu=5.0, flux_bot=0.05, bcs=bcs, theta_bcs=(bcs[0], "periodic", "noflux"), precision=prec)
    a, b = (AnelasticSimulation(g, isothermal_reference(n[2], 100.0, 2), **kw) for _ in range(2))
    rng = np.random.default_rng(sum(n))
    dt = np.float32 if prec else np.float64
    start = [np.asfortranarray(rng.standard_normal(g.storage).astype(dt)) for _ in range(4)]
    start[3] += dt(300)
    for sim in (a, b):
        for f, x in zip((sim.u, sim.v, sim.w, sim.theta), start):
            f.upload(x)
    h = 2.0
    a.step_rk3(h)
    fields = (b.u, b.v, b.w, b.theta)
    b.step(h)
    for ca in (0.75, 1.0 / 3.0):
        b.step(h)
        for f, x in zip(fields, start):
            f.upload(np.asfortranarray((ca * x.astype(np.float64) + (1 - ca) * f.download().astype(np.float64)).astype(dt)))
    for f, r in zip((a.u, a.v, a.w, a.theta, a.p), fields + (b.p,)):
        assert rel_err(f.download(), r.download()) <= tol
