"""The coarsest level's solve in FP32, in each of its forms: 1 to 4 cells of a
colour per thread (4, for 3073 to 4096 slots of a colour, is FP32's alone) and a
launch per half-sweep past them, on an open and on a coefficient operator.

Odd extents give one-level hierarchies: one iteration of the CG is x = α z with z
the 50 red-black sweeps of r, against the oracle's FP64 levels. A half-sweep is a
weighted mean of at most six neighbours (norm <= 1) in about 10 roundings of
2^-24, so 100 of them add at most 6e-5 of the largest value, and α, a ratio of
FP64 sums over z, as much again. A cell left out, or a neighbour of another cell,
shows at 1e-2.
"""
import ctypes

import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu

# extents, slots of a colour
SIZES = [((5, 4, 3), 36), ((15, 13, 9), 936), ((25, 17, 9), 1989), ((25, 17, 11), 2431), ((33, 17, 11), 3179),
         ((33, 17, 13), 3757), ((1, 61, 61), 3721), ((33, 17, 17), 4913)]


@pytest.mark.parametrize("coeff", [False, True])
@pytest.mark.parametrize("n,slots", SIZES)
def test_one_level(hip, orc, n, slots, coeff):
    assert (n[0] + 1) // 2 * n[1] * n[2] == slots
    rng = np.random.default_rng(sum(n))
    cs = None
    if coeff:
        cs = [np.asfortranarray(rng.uniform(0.2, 1.0, tuple(m + (a == q) for a, m in enumerate(n)))) for q in range(3)]
        for q, a in enumerate(cs):  # the walls' faces are closed
            a[tuple(slice(None) if s != q else [0, -1] for s in range(3))] = 0.0
    b = np.asfortranarray(rng.standard_normal(n))
    L = orc.lib()
    h = L.orc_mg_create(*n, 1.0, 1.3, 0.7, *[orc.BCS["neumann"]] * 3, *([None] * 3 if cs is None else map(orc.ptr, cs)),
                        None, 2, 2, 4, 0, 1.0)
    assert L.orc_mg_levels(h) == 1
    x = np.zeros(n, order="F")
    it, res, bn = ctypes.c_int(), ctypes.c_double(), ctypes.c_double()
    L.orc_mgpcg_solve(h, orc.ptr(x), orc.ptr(b), 1e-30, 1, ctypes.byref(it), ctypes.byref(res), ctypes.byref(bn))
    L.orc_mg_destroy(h)
    s = hip.MGPreconditionedCG(n, (1.0, 1.3, 0.7), bcs=("neumann",) * 3, coeff=cs, tol=1e-30, maxit=1, vcycle="f32")
    got = hip.solve_interior(s, b)
    assert hip.solver_stats(s)[0] == it.value == 1
    assert rel_err(got, x) < 1.2e-4
