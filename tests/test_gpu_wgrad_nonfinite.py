"""Infinities in one channel stay in that channel's weight gradients.

One last-level convolution (dec2_0, 16 channels to 16) is driven so that one
channel of its input, or of the gradient of its output, is infinite in every
voxel and everything else is finite; the other channels' gradients have to be
those of the same network with a large finite number in its place, up to the
order of the atomic sums."""
import numpy as np
import pytest

import test_unet

pytestmark = pytest.mark.gpu

LEVELS, C0 = 2, 16
Q = 5  # the channel
BIG = np.float32(3.4e38)  # infinite in BF16, and in FP32 once multiplied by 10


@pytest.mark.parametrize("where", ["input", "gradient"])
@pytest.mark.parametrize("dims", [(2, 2, 2), (20, 70, 6), (36, 12, 34)])
def test_other_channels_are_untouched(qesmc, where, dims):
    import unet_oracle as U

    dx, dy, dz = dims
    layers, head, n = U.layout(LEVELS, C0)
    at = {name: (cin, cout, woff, boff) for name, cin, cout, woff, boff in layers}
    cin, cout, woff, boff = at["dec2_0"]
    assert cin == cout == C0
    x = test_unet.rand_input((dz, dy, dx), 41)
    gy = np.random.default_rng(42).standard_normal((dz, dy, dx)).astype(np.float32)
    gy[np.abs(gy) < 0.1] = 0.1  # no product with the infinite weight is 0 * inf
    out = []
    for big in (np.float32(1e30), BIG):
        p = test_unet.he_params(LEVELS, C0, 40).astype(np.float32)
        if where == "input":
            # channel Q of E (dec1_0's output) is its bias; dec2_0 weighs it so that every output passes its ReLU
            dcin, dcout, dw, db = at["dec1_0"]
            p[dw:dw + 27 * dcin * dcout].reshape(dcout, -1)[Q] = 0.0
            p[db + Q] = big
            p[woff:woff + 27 * cin * cout].reshape(cout, 27, cin)[:, :, Q] = 1e-3
        else:
            # channel Q of the gradient of dec2_0's output, which is positive everywhere
            p[boff:boff + cout] = 1e6
            p[head + Q] = big
        net = qesmc.UNet(dx, dy, dz, levels=LEVELS, base_channels=C0, seed=7)
        net.set_params(p)
        net.forward(x)
        g = gy if where == "input" else gy * np.float32(100.0)
        out.append(net.backward(g)[woff:woff + 27 * cin * cout].reshape(cout, 27, cin).copy())
        net.close()
    axis = 2 if where == "input" else 0
    finite, infinite = out
    others = [np.delete(a, Q, axis=axis) for a in out]
    assert np.isfinite(others[0]).all() and np.abs(others[0]).max() > 0
    assert not np.isfinite(np.take(infinite, Q, axis=axis)).any()
    # up to 34 work-groups' sums in any order: their roundings, 2^-24 each in either run
    assert np.isfinite(others[1]).all()
    assert np.abs(others[1] - others[0]).max() <= 34 * 2.0 ** -23 * np.abs(others[0]).max()
