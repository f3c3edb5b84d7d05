"""The tiled terrain tendencies at the edges of their blocks, against the oracle.

FP64: a few tens of roundings per flux and densities carried over at most 32
levels by their ratio (2 roundings a half level), against the largest
tendency: 1e-12, as for the other sizes. FP32 fluxes: the bound stated for
them elsewhere, 1e-4. A flux taken from the wrong cell shows at 0.1. Sizes:
columns and rows one past, one short of and below the block's 64 x 4, a last
block of one cell, and chunks of 1, 2 and 17 levels with remainders (32 in
test_gpu_long_chunks.py).
"""
import numpy as np
import pytest

from helpers import rel_err
from test_gpu_terrain_core import LID, _random_state, _setup, _up

pytestmark = pytest.mark.gpu

SIZES = [(6, 6, 8), (63, 5, 13), (65, 9, 37), (130, 7, 50), (64, 72, 33), (192, 160, 67)]


@pytest.mark.parametrize("scheme,flux,tol", [("centered", "f64", 1e-12), ("weno_z5", "f64", 1e-12), ("weno_z5", "f32", 1e-4)])
@pytest.mark.parametrize("n", SIZES)
def test_tendencies(hip, orc, n, scheme, flux, tol):
    g, og, sim, core, tg = _setup(hip, orc, scheme=scheme, flux=flux, n=n)
    u, v, w, th = _random_state(og, core, 20, U=10.0)
    ref = core.tendencies(u, v, w, th)
    I, H = og.interior, og.H
    if flux == "f32":  # its form less θ_c·(B u)/(ρ̄J), added back
        J = (LID - tg.plane[H:H + og.Nx, H:H + og.Ny]) / LID
        ref[3][I] += th[I] * core.divergence(u, v, w) / (core.density(0)[I] * J[:, :, None])
    got = sim.tendencies([_up(a) for a in (u, v, w, th)])
    for a, b, name in zip(got, ref, ("tu", "tv", "tw", "ttheta")):
        err = rel_err(a.download()[I], b[I])
        assert err <= tol, (name, err)
