"""The marching kernels at the short chunks their rule picks on small grids: one
level per block on the smallest, up to 6 in the tile and brick kernels and 3 in
the limited one, with a shorter last chunk, against the CPU oracle (the longest
chunks: test_gpu_long_chunks.py). The values of a face do not depend on the
chunk it is computed in, so the tolerance is the parity tests' (FP64 roundings
of a fused multiply-add, 1e-12 relative)."""
import numpy as np
import pytest

from helpers import rand_storage, rel_err

pytestmark = pytest.mark.gpu

TOL64 = 1e-12
SIZES = [(8, 6, 5), (66, 9, 7), (64, 40, 29), (130, 72, 31), (190, 88, 37)]


@pytest.mark.parametrize("scheme,H", [("weno_z5", 3), ("weno_z7", 4)])
@pytest.mark.parametrize("N", SIZES)
def test_advection_at_every_chunk_length(hip, orc, N, scheme, H):
    g, og = (G(N, (3.0, 1.0, 2.0), halo=H) for G in (hip.Grid, orc.Grid))
    bcs = ("periodic",) * 3
    u, v, w, phi = (rand_storage(og.storage, 7 + q) for q in range(4))
    for a, loc in ((u, 1), (v, 2), (w, 3), (phi, 0)):
        orc.fill_halos(og, a, loc, bcs)
    dev = [hip.DeviceArray.from_numpy(a) for a in (u, v, w, phi)]
    I = og.interior
    ref = orc.advect_momentum(og, og.zeros(), og.zeros(), og.zeros(), u, v, w, scheme)
    out = [g.field() for _ in range(3)]
    hip.advection_scheme(scheme, g).momentum(*out, *dev[:3])
    for a, b in zip(out, ref):
        assert rel_err(a.download()[I], b[I]) <= TOL64
    t = g.field()
    hip.advection_scheme(scheme, g)(t, *dev)
    assert rel_err(t.download()[I], orc.advect_scalar(og, og.zeros(), u, v, w, phi, scheme)[I]) <= TOL64
    phi = np.abs(phi)
    t = g.field()
    hip.advect_positive(g, t, *dev[:3], hip.DeviceArray.from_numpy(phi), 0.01, scheme=scheme, accumulate=False)
    ref = orc.advect_positive(og, og.zeros(), u, v, w, phi, 0.01, scheme=scheme, accumulate=False)
    assert rel_err(t.download()[I], ref[I]) <= TOL64
