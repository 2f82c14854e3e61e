"""Large copies between the caller's arrays and the device come back byte for
byte: at the sizes where the pinned slots take over (8 MiB towards the host,
128 MiB towards the device), odd lengths, and from two threads at once, one
of which finds the slots lent."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def round_trip(Q, ncx, ncy, ncz, seed, times=1):
    with Q.Context(0) as c:
        c.set_city(ncx, ncy, 1.0, Q.dz_uniform(ncz, 1.0), [], (1, 4.0, 10.0, 0.5, 250.0))
        rng = np.random.default_rng(seed)
        for _ in range(times):
            lam = rng.integers(0, 1 << 32, c.city.ncell, dtype=np.uint32).view(np.float32)
            c.set_lambda(lam)
            assert np.array_equal(c.get_lambda().view(np.uint32), lam.view(np.uint32))


# cells (ncz + 1 layers): 2 Mi is 8 MiB, 32 Mi is 128 MiB
@pytest.mark.parametrize("shape", [(128, 128, 127), (127, 127, 129), (129, 131, 126), (512, 512, 127), (513, 511, 129)])
def test_round_trip(qesmc, shape):
    round_trip(qesmc, *shape, seed=sum(shape))


def test_velocity_of_a_resident_inflow(qesmc):
    """Three arrays in one call: u, v, w of a run without iterations from
    lambda = 0 are u0, v0, w0 off the solid cells."""
    with qesmc.Context(0) as c:
        c.set_city(200, 150, 1.0, qesmc.dz_uniform(40, 1.0), [], (1, 4.0, 10.0, 0.5, 250.0))
        n = c.city.nface
        rng = np.random.default_rng(1)
        u0, v0, w0 = (rng.standard_normal(n).astype(np.float32) for _ in range(3))
        c.set_inflow(u0, v0, w0)
        c.run(itermax=0)
        for got, want in zip(c.get_velocity(), (u0, v0, w0)):
            assert np.array_equal(got, want)


def test_two_threads(qesmc):
    errors = []

    def go(seed):
        try:
            round_trip(qesmc, 260, 260, 60, seed, times=6)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=go, args=(s,)) for s in (1, 2, 3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
