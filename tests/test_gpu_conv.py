"""The U-Net's convolution at the edges of its bricks: 16 voxels along x by 8
rows by 4 planes, or, where all channels are staged, 4 x 4 down to 1 x 2."""
import numpy as np
import pytest

import test_unet

pytestmark = pytest.mark.gpu


# volumes below and above 1024 bricks of 8 x 8 x 4 (the two orders of products), each with a
# ragged last brick in x, y and z on every level
@pytest.mark.parametrize("levels,c0,dims", [(2, 16, (2, 2, 2)), (2, 16, (20, 70, 6)), (2, 16, (200, 52, 36)),
                                            (3, 32, (36, 20, 12)), (2, 32, (136, 76, 60)), (4, 16, (56, 40, 24))])
def test_tile_edges(qesmc, levels, c0, dims):
    """Forward and gradients against the oracle, with the bounds that hold for
    every other size."""
    test_unet.test_device_forward_backward_match_oracle(qesmc, levels, c0, dims)


def test_planes_past_31_bits(qesmc):
    """A corner of a volume whose six planes of 96 channels take more than 2 GiB
    against the same corner cut out, large enough for the same order of
    products on both levels: equal bits 16 or more voxels from the cut
    (the network sees 10), and equal gradients but for the order of their sums."""
    levels, c0, dx, dy, dz, c = 2, 32, 2048, 1024, 2, 512
    rng = np.random.default_rng(31)
    p = test_unet.he_params(levels, c0, 32).astype(np.float32)
    corner = test_unet.rand_input((dz, c, c), 33)
    g = np.zeros((dz, c, c), np.float32)
    g[:, 384:, 384:] = rng.standard_normal((dz, c - 384, c - 384))
    out = []
    for nx, ny in ((c, c), (dx, dy)):
        net = qesmc.UNet(nx, ny, dz, levels=levels, base_channels=c0, seed=7)
        net.set_params(p)
        x = np.zeros((dz, ny, nx, 8), np.float32)
        x[:, -c:, -c:] = corner
        gg = np.zeros((dz, ny, nx), np.float32)
        gg[:, -c:, -c:] = g
        y = net.forward(x)[:, -c:, -c:].copy()
        out.append((y, net.backward(gg)))
        net.close()
    (ya, ga), (yb, gb) = out
    assert np.abs(ya).max() > 0.1
    assert np.array_equal(ya[:, 16:, 16:], yb[:, 16:, 16:])
    assert np.linalg.norm(ga - gb) <= 1e-4 * np.linalg.norm(ga)
