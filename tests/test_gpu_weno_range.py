"""WENO-Z5 and Z7 up to the end of FP64's range, against the oracle's form from
the values with one division per ratio.

The indicators are squares of the variation, and FP64 holds a square up to 1e308;
the products of two or three of them, in place of a division per ratio, end at
1e77 and 1e51 unless they are scaled. Scales on both sides of both ends, and
a jump of such a scale beside a smaller field or a flat one, where one product
holds small and large factors: the ratio there is the square of the scale, and its
own square has to be finite for the weights to be. 1e-12 as at the ordinary scales
(a few tens of roundings); a form that lost the range gives NaN.
"""
import numpy as np
import pytest

from helpers import rel_err
from test_gpu_weno_z import _case

pytestmark = pytest.mark.gpu

# 2^166 is 9e49, 2^249 1e75: the unscaled products' ends (three and two indicators)
SCALES = [133, 149, 166, 230, 249, 260, 330, 400, 480]


@pytest.mark.parametrize("scheme", ["weno_z5", "weno_z7"])
@pytest.mark.parametrize("e", SCALES)
def test_noise(hip, orc, e, scheme):
    got, ref = _case(orc, hip, lambda rng, s: np.asfortranarray(2.0**e * rng.standard_normal(s)), scheme)
    assert np.isfinite(ref).all() and np.abs(ref).max() > 2.0**e
    assert rel_err(got, ref) < 1e-12


@pytest.mark.parametrize("scheme", ["weno_z5", "weno_z7"])
@pytest.mark.parametrize("e", [60, 120, 180, 240])
def test_small_beside_large(hip, orc, e, scheme):
    def phi(rng, s):
        a = rng.standard_normal(s)
        a[s[0] // 2:] *= 2.0**e
        return np.asfortranarray(a)
    got, ref = _case(orc, hip, phi, scheme)
    assert np.isfinite(ref).all()
    # each half at its own scale, the stencils across the jump left to the large one's
    # (an unupwinded x-stencil reaches four cells; the fields are periodic)
    half = ref.shape[0] // 2
    assert rel_err(got, ref) < 1e-12
    assert rel_err(got[5:half - 5], ref[5:half - 5]) < 1e-12


@pytest.mark.parametrize("scheme", ["weno_z5", "weno_z7"])
@pytest.mark.parametrize("e", [0, 150, 200, 240, 300, 480])
def test_pulses(hip, orc, e, scheme):
    # jumps of one size on a flat field: equal indicators (τ = 0) beside vanishing
    # ones, whose product underflows against the large ones' squares. The
    # reference's own weights overflow where a ratio passes 1e154 (its squares):
    # its finite values are compared
    def phi(rng, s):
        a = np.zeros(s)
        a[::3] = 1.0
        a[:, ::4] += 1.0
        a[:, :, ::5] = 2.0
        return np.asfortranarray(2.0**e * a)
    with np.errstate(invalid="ignore"):
        got, ref = _case(orc, hip, phi, scheme)
    ok = np.isfinite(ref)
    assert ok.any() and np.isfinite(got[ok]).all()
    assert rel_err(got[ok], ref[ok]) < 1e-12


@pytest.mark.parametrize("scheme", ["weno_z5", "weno_z7"])
@pytest.mark.parametrize("e", [100, 200, 400])
def test_limited(hip, orc, e, scheme):
    n, H = (70, 21, 13), 4
    g, og = hip.Grid(n, (3.0, 1.0, 2.0), halo=H), orc.Grid(n, (3.0, 1.0, 2.0), halo=H)
    rng = np.random.default_rng(4)
    vel = []
    for loc in (orc.FX, orc.FY, orc.FZ):
        a = np.asfortranarray(rng.uniform(-1, 1, og.storage))
        orc.fill_halos(og, a, loc, ("periodic",) * 3)
        vel.append(a)
    f = np.asfortranarray(2.0**e * np.abs(rng.standard_normal(og.storage)))
    orc.fill_halos(og, f, orc.CC, ("periodic",) * 3)
    ref = orc.advect_positive(og, og.zeros(), *vel, f, 0.01, scheme=scheme, accumulate=False)
    t = g.field()
    up = hip.DeviceArray.from_numpy
    hip.advect_positive(g, t, *[up(a) for a in vel], up(f), 0.01, scheme=scheme, accumulate=False)
    I = og.interior
    assert np.isfinite(ref[I]).all() and rel_err(t.download()[I], ref[I]) < 1e-12


@pytest.mark.parametrize("scheme", ["weno_z5", "weno_z7"])
@pytest.mark.parametrize("e,half", [(0, False), (166, False), (330, False), (480, False), (120, True), (240, True),
                                    (440, True)])
def test_exponent_one(hip, orc, e, half, scheme):
    """p = 1, whose weights take the ratios themselves: small beside large up to 2^440."""
    n, H = (70, 21, 13), 4
    g, og = hip.Grid(n, (3.0, 1.0, 2.0), halo=H), orc.Grid(n, (3.0, 1.0, 2.0), halo=H)
    rng = np.random.default_rng(5)
    f = [np.asfortranarray(rng.standard_normal(og.storage)) for _ in range(4)]
    f[3][og.storage[0] // 2 if half else 0:] *= 2.0**e
    for a, loc in zip(f, (orc.FX, orc.FY, orc.FZ, orc.CC)):
        orc.fill_halos(og, a, loc, ("periodic",) * 3)
    ref = orc.advect_scalar(og, og.zeros(), *f, scheme, p=1)[og.interior]
    t = g.field()
    hip.advection_scheme(scheme, g, p=1)(t, *[hip.DeviceArray.from_numpy(a) for a in f])
    got = t.download()[og.interior]
    assert np.isfinite(ref).all() and rel_err(got, ref) < 1e-12
    if half:
        m = n[0] // 2
        assert rel_err(got[5:m - 5], ref[5:m - 5]) < 1e-12
