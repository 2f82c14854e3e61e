"""Copies through the pinned slots, once these are there, come back byte for
byte at the sizes where they take over, at odd lengths, and from several
threads of which one has them at a time."""
import threading

import pytest

import test_gpu_copy

pytestmark = pytest.mark.gpu


@pytest.fixture
def slots(qesmc):
    """A context whose copies have made the slots, and keep them."""
    with qesmc.Context(0) as c:
        c.set_city(300, 300, 1.0, qesmc.dz_uniform(100, 1.0), [], (1, 4.0, 10.0, 0.5, 250.0))
        c.run(itermax=0)
        c.get_velocity()  # 110 MB
        yield


@pytest.mark.parametrize("shape", [(128, 128, 127), (127, 127, 129), (129, 131, 126), (200, 150, 100)])
def test_round_trip(qesmc, slots, shape):
    test_gpu_copy.round_trip(qesmc, *shape, seed=sum(shape), times=2)


def test_velocity_of_a_resident_inflow(qesmc, slots):
    test_gpu_copy.test_velocity_of_a_resident_inflow(qesmc)


def test_threads(qesmc, slots):
    errors = []

    def go(seed):
        try:
            test_gpu_copy.round_trip(qesmc, 200, 200, 60, seed, times=6)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=go, args=(s,)) for s in (1, 2, 3, 4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
