"""The U-Net's weight and bias gradients at the sizes where their 32-voxel row
segments and row chunks can go wrong: axes of one voxel at the coarsest level,
one past and one short of a segment, several segments, rows past one chunk,
and one and two input channels. Against the CPU network oracle with BF16
rounding at the same points, per layer, at the tolerance stated for the
network's gradients (BF16 ties carried through ten layers: 5e-2 relative L2).
Blocks of several tasks, longer row chunks and the sums to FP32 rounding:
test_gpu_weight_gradient.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPEC = [(16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (96, 32), (32, 32), (48, 16), (16, 16)]


@pytest.mark.parametrize("shape,inc", [((4, 4, 4), 2), ((28, 4, 8), 1), ((36, 12, 4), 2), ((64, 36, 8), 2),
                                       ((132, 20, 4), 1)])
def test_layer_gradients(hip, orc, shape, inc):
    from aeolus_hip.fields import DeviceArray
    from aeolus_hip.learned import UNet
    rng = np.random.default_rng(sum(shape))
    net = UNet(shape, in_channels=inc, seed=3)
    p = net.params()
    p[-17:] += 0.1 * rng.standard_normal(17).astype(np.float32)
    net.set_params(p)
    src, tgt = rng.standard_normal(shape), rng.standard_normal(shape)
    mask = (rng.random(shape) > 0.3).astype(np.float64) if inc == 2 else None
    dev = [None if a is None else DeviceArray.from_numpy(a) for a in (src, tgt, mask)]
    loss, g = net.gradients(*dev)
    again = net.gradients(*dev)[1]
    assert np.array_equal(g, again)  # the sums run in a fixed order
    loss_ref, ref = orc.unet_gradients(p, src, tgt, mask, bf16=True)
    assert abs(loss - loss_ref) < 1e-3 * loss_ref
    off = 0
    for li, (cin, cout) in enumerate([(inc, 16)] + SPEC):
        for n in (27 * cin * cout, cout):
            a, b = g[off:off + n], ref[off:off + n]
            assert np.linalg.norm(a - b) < 5e-2 * max(np.linalg.norm(b), 1e-30), (li, n)
            off += n
