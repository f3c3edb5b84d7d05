"""The weight and bias gradients of one convolution alone, against the float64 sum
over the kernel's own BF16 inputs: where blocks take several tasks (a barrier
before the next task's rows, the row slots and buffers used again, the sums
kept across tasks), in row chunks of 8, 16 and 32, in one and in several channel
slices.

The products of two BF16 numbers are exact in FP32, and a block adds them into
FP32 sums 32 voxels at a time: s steps of a sum add at most (s + 32) roundings
of 2^-24 (the unit may truncate: 2^-23) of the sum of the magnitudes, and the
partials are added in float64. Rows left out, added twice or read from another
task's slot show at 1e-3 of the same measure.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bf16(rng, shape):
    """Random BF16 values: (their bits, the same as float64)."""
    bits = (rng.standard_normal(shape).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    return bits, (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def _reference(x, dy):
    """dW[tap][c][n] and db[n]: x and y periodic, z zero-padded (arrays [z, y, x, channel])."""
    nz, c, n = x.shape[0], x.shape[-1], dy.shape[-1]
    dw = np.empty((27, c, n))
    d = dy.reshape(-1, n)
    for t in range(27):
        sx, sy, sz = t % 3 - 1, t // 3 % 3 - 1, t // 9 - 1
        s = np.zeros_like(x)
        s[max(0, -sz):nz - max(0, sz)] = x[max(0, sz):nz - max(0, -sz)]
        dw[t] = np.roll(s, (-sy, -sx), (1, 2)).reshape(-1, c).T @ d
    return dw, d.sum(0)


# layer, extents, rows of a task, more tasks than blocks
CASES = [((16, 16), (36, 72, 136), 32, True), ((8, 16), (33, 41, 208), 32, True), ((48, 16), (36, 72, 136), 32, True),
         ((16, 32), (36, 72, 136), 32, True), ((32, 32), (31, 40, 400), 32, True), ((32, 64), (36, 72, 68), 32, True),
         ((96, 32), (36, 72, 45), 32, True), ((64, 64), (36, 72, 34), 32, True),
         ((16, 16), (36, 72, 60), 16, False), ((64, 64), (36, 40, 22), 16, False), ((64, 64), (8, 8, 4), 8, False),
         ((32, 64), (70, 5, 3), 8, False), ((16, 32), (1, 1, 1), 8, False)]


@pytest.mark.parametrize("layer,n,rows,many", CASES)
def test_against_float64(hip, layer, n, rows, many):
    from aeolus_hip import _lib as L
    lib = L.init()
    rng = np.random.default_rng(sum(n) + layer[0])
    (xb, x), (db, dy) = (_bf16(rng, n[::-1] + (c,)) for c in layer)
    dw, bias = np.empty((27,) + layer, np.float32), np.empty(layer[1], np.float32)
    ptr = [ctypes.c_void_p() for _ in range(4)]
    for p, a in zip(ptr, (xb, db, dw, bias)):
        L.check(lib.aeo_malloc(ctypes.byref(p), a.nbytes))
    for p, a in zip(ptr, (xb, db)):
        L.check(lib.aeo_memcpy_h2d(p, a.ctypes.data_as(ctypes.c_void_p), a.nbytes))
    plan = (ctypes.c_int * 3)()
    L.check(lib.aeo_conv3_weight_gradient(*layer, *n, *ptr, plan))
    for p, a in zip(ptr[2:], (dw, bias)):
        L.check(lib.aeo_memcpy_d2h(a.ctypes.data_as(ctypes.c_void_p), p, a.nbytes))
    for p in ptr:
        L.check(lib.aeo_free(p))
    assert plan[0] == rows and (plan[1] > plan[2]) == many
    steps = -(-plan[1] // plan[2]) * rows
    tol = (steps + 32) * 2.0**-23
    ref, mag = _reference(x, dy), _reference(np.abs(x), np.abs(dy))
    for got, r, m in zip((dw, bias), ref, mag):
        assert np.abs(m).min() > 0 or n[2] == 1
        assert np.all(np.abs(got - r) <= tol * m + 1e-30)


def test_bad_arguments(hip):
    from aeolus_hip import _lib as L
    lib = L.init()
    p = ctypes.c_void_p(256)  # never read: refused before any launch
    assert lib.aeo_conv3_weight_gradient(16, 24, 4, 4, 4, p, p, p, p, None) != 0
    assert lib.aeo_conv3_weight_gradient(16, 16, 0, 4, 4, p, p, p, p, None) != 0
    assert lib.aeo_conv3_weight_gradient(16, 16, 2048, 2048, 64, p, p, p, p, None) != 0
    assert lib.aeo_conv3_weight_gradient(16, 16, 4, 4, 4, None, p, p, p, None) != 0
