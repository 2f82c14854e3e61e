"""Pinned arrays of the caller's come back byte for byte, alone and beside
pageable ones, in both directions, above and below the sizes where pageable
arrays take the library's slots."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def pointer(a):
    return C.cast(a.data_ptr() if isinstance(a, torch.Tensor) else a.ctypes.data, C.POINTER(C.c_float))


@pytest.mark.parametrize("shape,pinned", [((40, 30, 20), (0, 1, 2)), ((400, 300, 120), (0, 1, 2)),
                                          ((400, 300, 120), (1,)), ((400, 300, 120), ())])
def test_velocity_of_a_pinned_inflow(qesmc, shape, pinned):
    """u, v, w of a run without iterations from lambda = 0 are u0, v0, w0 off
    the solid cells."""
    ncx, ncy, ncz = shape
    with qesmc.Context(0) as c:
        c.set_city(ncx, ncy, 1.0, qesmc.dz_uniform(ncz, 1.0), [], (1, 4.0, 10.0, 0.5, 250.0))
        n = c.city.nface
        gen = torch.Generator().manual_seed(n)

        def arrays(fill):
            out = [torch.empty(n, pin_memory=True) if q in pinned else torch.empty(n) for q in range(3)]
            for a in out:
                fill(a)
            return out

        inflow = arrays(lambda a: a.copy_(torch.randn(n, generator=gen)))
        got = arrays(lambda a: a.fill_(7.0))
        L = qesmc.lib()
        assert L.qesmc_set_inflow(c._h, *[pointer(a) for a in inflow]) == qesmc.OK
        c.run(itermax=0)
        assert L.qesmc_get_velocity(c._h, *[pointer(a) for a in got]) == qesmc.OK
        for a, b in zip(got, inflow):
            assert np.array_equal(a.numpy(), b.numpy())
