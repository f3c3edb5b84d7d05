"""The terrain core's halos at odd sizes, rows and columns fewer than the halo is
wide excepted (the periodic images need N >= H), bit for bit up to the
diagnosed w faces (one expression, within 1e-15)."""
import numpy as np
import pytest

from helpers import rand_storage, rel_err
from test_gpu_terrain_core import _setup, _up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(4, 4, 4), (3, 7, 5), (61, 5, 9), (130, 43, 6)])
def test_halos(hip, orc, n):
    g, og, sim, core, _ = _setup(hip, orc, n=n)
    f = [rand_storage(og.storage, 10 + s) for s in range(4)]
    dev = [_up(a) for a in f]
    sim.fill_halos(dev)
    core.fill_halos(*f)
    for a, b in zip(dev, f):
        assert rel_err(a.download(), b) <= 1e-15
