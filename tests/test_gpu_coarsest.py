"""The coarsest level's solve in one workgroup against the CPU oracle.

Odd extents give one-level hierarchies, so one cycle is 50 red-black sweeps
of the whole grid. The sizes reach every form of the solve: 1, 2 and 3 cells
of a colour per thread, the form that reads its weights from memory (rows of
one cell), and a level past the registers, which takes a launch per
half-sweep. Neumann axes: no cell has a neighbour of its own colour.
"""
import ctypes

import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu

SIZES = [(3, 3, 3), (5, 4, 3), (15, 13, 9), (25, 17, 9), (25, 17, 11), (1, 61, 61), (33, 17, 11)]


def _coeffs(N, seed):
    rng = np.random.default_rng(seed)
    cs = [np.asfortranarray(rng.uniform(0.2, 1.0, tuple(n + (a == q) for a, n in enumerate(N)))) for q in range(3)]
    c = [n // 2 for n in N]  # one fully blocked cell
    for q, a in enumerate(cs):
        for e in (0, 1):
            i = list(c)
            i[q] += e
            a[tuple(i)] = 0.0
    return cs, tuple(c)


@pytest.mark.parametrize("blocked", [False, True])
@pytest.mark.parametrize("N", SIZES)
def test_one_level_cycle(hip, orc, N, blocked):
    cs, cell = _coeffs(N, 5)
    src = np.asfortranarray(np.random.default_rng(6).normal(size=N))
    if blocked:
        src[cell] = 0.0
        src -= src.sum() / (src.size - 1)
        src[cell] = 0.0
    else:
        cs = None
    L = orc.lib()
    h = L.orc_mg_create(*N, 1.0, 1.3, 0.7, *[orc.BCS["neumann"]] * 3, *([None] * 3 if cs is None else map(orc.ptr, cs)),
                        None, 2, 2, 4, 0, 1.0)
    assert L.orc_mg_levels(h) == 1
    ref = np.zeros(N, order="F")
    rel = ctypes.c_double()
    L.orc_mg_solve(h, orc.ptr(ref), orc.ptr(src), 1e-30, 1, ctypes.byref(rel))
    L.orc_mg_destroy(h)
    s = hip.MultigridPoissonSolver(N, (1.0, 1.3, 0.7), bcs=("neumann",) * 3, coeff=cs, tol=1e-30, maxcycles=1)
    x = hip.solve_interior(s, src)
    # a sweep is a weighted mean of at most six neighbours (norm <= 1), so the 100
    # half-sweeps add at most 100 roundings of about 10 eps each to the values
    assert rel_err(x, ref) < 100 * 10 * np.finfo(np.float64).eps * 5
