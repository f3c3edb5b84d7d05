"""WENO-Z5 and Z7 from differences, with the weights' ratios from one reciprocal
per three or two (FP64), at the ends of their range, against the oracle's form from the values.

Each of the two forms rounds the smoothness indicators and candidates a few
times (about 10 roundings of 1.1e-16 of the largest stencil value each, times
the three directions and the flux difference), so 1e-12 of the largest
tendency holds at every scale; the scales are those where the indicators
vanish against ε², where they are far above it, and where the product of the
three is far up FP64's range (1e240). They are powers of two, so that the steps
stay exact: where two indicators are equal and the third is 0, τ is 0, and a
rounded step would make it noise divided by ε² = 5e-32, of any size in either
form.
"""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu


def _case(orc, hip, phi, scheme, n=(70, 21, 13), H=4):
    g, og = hip.Grid(n, (3.0, 1.0, 2.0), halo=H), orc.Grid(n, (3.0, 1.0, 2.0), halo=H)
    rng = np.random.default_rng(3)
    up = hip.DeviceArray.from_numpy
    vel = []
    for loc in (orc.FX, orc.FY, orc.FZ):
        a = np.asfortranarray(rng.standard_normal(og.storage))
        orc.fill_halos(og, a, loc, ("periodic",) * 3)
        vel.append(a)
    f = phi(rng, og.storage)
    orc.fill_halos(og, f, orc.CC, ("periodic",) * 3)
    ref = orc.advect_scalar(og, og.zeros(), *vel, f, scheme)
    t = up(og.zeros())
    hip.advection_scheme(scheme, g)(t, *[up(a) for a in vel], up(f))
    return t.download()[og.interior], ref[og.interior]


@pytest.mark.parametrize("scheme", ["weno_z5", "weno_z7"])
@pytest.mark.parametrize("scale", [2.0**-83, 2.0**-53, 1.0, 2.0**40, 2.0**133])
@pytest.mark.parametrize("kind", ["noise", "steps", "offset"])
def test_scales(hip, orc, scale, kind, scheme):
    def phi(rng, s):
        a = rng.standard_normal(s)
        if kind == "steps":  # flat stretches (every indicator 0) and jumps
            a = np.round(a / 2)
        if kind == "offset":  # a mean far above the variation
            a = 300.0 + 0.1 * a
        return np.asfortranarray(scale * a)
    got, ref = _case(orc, hip, phi, scheme)
    assert np.abs(ref).max() > 0 and rel_err(got, ref) < 1e-12


@pytest.mark.parametrize("scheme", ["weno_z5", "weno_z7"])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_a_bad_cell_stays_in_its_stencils(hip, orc, bad, scheme):
    def phi(rng, s):
        a = np.asfortranarray(rng.standard_normal(s))
        a[30, 10, 8] = bad
        return a
    got, ref = _case(orc, hip, phi, scheme)
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    ok = np.isfinite(ref)
    assert rel_err(got[ok], ref[ok]) < 1e-12
