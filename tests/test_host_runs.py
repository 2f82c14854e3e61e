"""What the library's host code decides, on the CPU: which kernels a call
launches, what it allocates, and what becomes of it when an allocation fails.

Each case runs in a process of its own against tests/cpp/hip_stand_in.cpp, a
stand-in for the HIP runtime whose kernels do nothing; what the kernels compute
is the GPU tests' business."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FLAT = (1, 4.0, 10.0, 0.5, 230.0)


class StandIn:
    """The stand-in's controls: allocations and launches since reset()."""

    def __init__(self, path):
        # under the runtime's own soname, so that the library finds it loaded
        self.lib = C.CDLL(path, mode=C.RTLD_GLOBAL)
        self.lib.stand_in_value.restype = C.c_longlong
        self.lib.stand_in_cost.argtypes = [C.c_char_p, C.c_double]
        self.lib.stand_in_fail_at.argtypes = self.lib.stand_in_fail_above.argtypes = [C.c_longlong]
        self.lib.stand_in_news.argtypes = [C.c_int, C.c_longlong]
        self.reset, self.fail_at, self.fail_above = (getattr(self.lib, "stand_in_" + n)
                                                     for n in ("reset", "fail_at", "fail_above"))

    def launches(self, kernel):
        return self.lib.stand_in_launches(kernel.encode())

    def grid(self, kernel):
        return self.lib.stand_in_grid(kernel.encode())

    def cost(self, kernel, us):
        self.lib.stand_in_cost(kernel.encode(), us)

    def news(self, fail_at=0):
        """Count this thread's C++ allocations; the fail_at-th fails."""
        self.lib.stand_in_news(1, fail_at)

    def value(self, what):
        return self.lib.stand_in_value(
            ("device_allocs", "host_allocs", "live", "news", "syncs", "graph_launches", "copied", "host_live").index(what))


def flat_city(Q, ncx, ncy, ncz):
    c = Q.Context(0)
    c.set_city(ncx, ncy, 2.0, Q.dz_uniform(ncz, 1.0), [], FLAT)
    return c


# 32.8 M cells: arrays beyond the 256 MB Infinity Cache, so AUTO is reported as FUSED
BEYOND = (640, 400, 127)
LAMBDA = 4 * 640 * 400 * 128  # bytes of the second lambda, at least


def case_auto_beyond_the_cache_without_memory(Q, S):
    """AUTO takes the colour passes, and says so, where the march's buffers
    cannot be had; an explicit FUSED is refused."""
    with flat_city(Q, *BEYOND) as c:
        c.run(itermax=2, path=Q.PATH_SPLIT)  # the convergence rows
        S.reset()
        S.fail_above(LAMBDA - 1)
        r = c.run(itermax=4)
        assert r["path"] == Q.PATH_SPLIT and r["tile_v"] in (1, 2, 4) and r["wg_per_cu"] > 0, r
        assert S.launches("k_sor_split") == 8 and S.launches("k_sor_march") == 0
        try:
            c.run(itermax=4, path=Q.PATH_FUSED)
            assert False, "FUSED without its buffers"
        except Q.QesmcError as e:
            assert e.code == Q.ERR_OOM
        S.reset()
        r = c.run(itermax=4)
        assert r["path"] == Q.PATH_FUSED and S.launches("k_sor_march") > 0 and S.launches("k_sor_split") == 0


def case_batch_with_a_member_without_memory(Q, S):
    """A member beyond the cache whose march buffers cannot be had sends the
    whole batch to the colour passes."""
    with flat_city(Q, 40, 30, 20) as a, flat_city(Q, *BEYOND) as b:
        for c in (a, b):
            c.run(itermax=2, path=Q.PATH_SPLIT)
        S.reset()
        S.fail_above(LAMBDA - 1)
        Q.run_batch([a, b], itermax=4, check_every=4, use_graph=False)
        assert S.launches("k_sor_batch") == 8 and S.launches("k_sor_march") == 0


def case_static_run_after_a_half_made_set(Q, S):
    """Whichever of the march's five buffers could not be had, a FUSED
    qesmc_run_static is refused and allocates nothing."""
    for nth in range(1, 6):
        with flat_city(Q, 40, 30, 20) as c:
            c.run(itermax=2, path=Q.PATH_SPLIT)
            S.fail_at(nth)
            c.run(itermax=2)
            S.reset()
            try:
                c.run_static(itermax=2, path=Q.PATH_FUSED)
                assert False, nth
            except Q.QesmcError as e:
                assert e.code == Q.ERR_STATE, (nth, e.code)
            assert S.value("device_allocs") == S.value("host_allocs") == 0, nth


def case_half_made_set_is_given_back(Q, S):
    """A run that cannot have all of the march's buffers keeps none of them,
    whether it goes on with the colour passes or is refused."""
    for nth in range(1, 6):
        with flat_city(Q, 40, 30, 20) as c:
            c.run(itermax=2, path=Q.PATH_SPLIT)
            before = S.value("live")
            S.fail_at(nth)
            assert c.run(itermax=2)["path"] == Q.PATH_SPLIT
            assert S.value("live") == before, nth
            S.fail_at(nth)
            try:
                c.run(itermax=2, path=Q.PATH_FUSED)
                assert False, nth
            except Q.QesmcError as e:
                assert e.code == Q.ERR_OOM
            assert S.value("live") == before, nth
            S.reset()
            c.run(itermax=2)
            assert S.launches("k_sor_march") > 0 and S.value("live") > before


def case_static_run_on_a_new_geometry(Q, S):
    """qesmc_run_static allocates nothing, on the device or the host, on its
    first march after a new geometry of the same size."""
    with flat_city(Q, 300, 40, 20) as c:
        c.run(itermax=2)
        for path in (Q.PATH_AUTO, Q.PATH_FUSED):
            c.set_city(300, 40, 2.0, Q.dz_uniform(20, 1.0), [], FLAT)
            S.reset()
            S.news()
            c.run_static(itermax=4, path=path)
            assert S.value("news") == S.value("device_allocs") == S.value("host_allocs") == 0, S.value("news")
            assert S.launches("k_pair_masks") == 1 and S.launches("k_sor_march") > 0


def refusing_each_allocation(Q, S, call):
    """call() once for every C++ allocation it makes, that one refused: it
    returns (a status, not an exception across the C interface)."""
    refused = 0
    for nth in range(1, 10000):
        S.news(fail_at=nth)
        try:
            call()
        except Q.QesmcError as e:
            assert e.code == Q.ERR_OOM, e.code
            refused += 1
        hit = S.value("news") >= nth
        S.news()
        if not hit:
            return refused
    assert False, "never done"


def case_no_host_memory_for_a_batch(Q, S):
    ctxs = [flat_city(Q, 30 + 5 * q, 40, 20) for q in range(3)]
    for kw in (dict(), dict(path=Q.PATH_SPLIT)):
        n = refusing_each_allocation(Q, S, lambda: Q.run_batch(ctxs, itermax=4, check_every=4, use_graph=True, **kw))
        assert n >= 3
        S.reset()
        Q.run_batch(ctxs, itermax=4, check_every=4, use_graph=False, **kw)  # as if nothing had happened
        assert S.launches("k_sor_march" if not kw else "k_sor_batch") > 0
    for c in ctxs:
        c.close()


def case_no_host_memory_for_a_copy(Q, S):
    """A large copy without the memory for its chunks or its threads."""
    with flat_city(Q, 200, 200, 60) as c:
        c.run(itermax=2)
        refusing_each_allocation(Q, S, c.get_velocity)
        refusing_each_allocation(Q, S, lambda: c.run(itermax=2))
        u, v, w = c.get_velocity()
        assert not u.any() and not v.any() and not w.any()


def tiles(r):
    return (r["tile_k"], r["tile_v"], r["wg_per_cu"])


def case_autotune_keeps_the_march_where_it_is_faster(Q, S):
    """The tuned tiling of the colour passes is kept and reported, and AUTO
    goes on marching: with tile fields 0 and with the tuned ones."""
    for dims, path in (((40, 30, 20), Q.PATH_SPLIT), (BEYOND, Q.PATH_FUSED)):
        with flat_city(Q, *dims) as c:
            S.cost("k_sor_split", 20.0)
            for iterations in (1, 20):
                best = Q.autotune(c, iterations=iterations)
                assert best.tile_k > 0 and best.tile_v > 0 and best.wg_per_cu > 0
                for p in (Q.default_params(itermax=10), best):
                    p.itermax = 10
                    S.reset()
                    r = c.run(p)
                    assert S.launches("k_sor_march") > 0 and S.launches("k_sor_split") == 0, iterations
                    assert r["path"] == path and (path == Q.PATH_FUSED or tiles(r) == tiles(vars_of(best)))
            if path == Q.PATH_SPLIT:  # another tiling, or a path, is still the caller's word
                for kw in (dict(tile_v=3 - min(best.tile_v, 2)), dict(tile_k=best.tile_k), dict(path=Q.PATH_SPLIT)):
                    S.reset()
                    c.run(itermax=10, **kw)
                    assert S.launches("k_sor_march") == 0 and S.launches("k_sor_split") == 20, kw


def vars_of(p):
    return {n: getattr(p, n) for n, _ in p._fields_}


def case_autotune_leaves_the_march_where_it_is_slower(Q, S):
    for dims in ((40, 30, 20), BEYOND):
        with flat_city(Q, *dims) as c:
            S.cost("k_sor_march", 1000.0)
            best = Q.autotune(c, iterations=20)
            for p in (Q.default_params(), best):
                p.itermax = 10
                S.reset()
                r = c.run(p)
                assert S.launches("k_sor_march") == 0 and S.launches("k_sor_split") == 20
                assert r["path"] == Q.PATH_SPLIT and tiles(r) == tiles(vars_of(best))
            # another grid has not been tuned
            c.set_city(50, 30, 2.0, Q.dz_uniform(20, 1.0), [], FLAT)
            S.reset()
            c.run(itermax=10)
            assert S.launches("k_sor_march") > 0


def case_results_tell_what_ran(Q, S):
    """qesmc_result.reserved: SOR iterations per launch, 0 for a launch per colour."""
    with flat_city(Q, 40, 30, 20) as a, flat_city(Q, 50, 30, 20) as b:
        for kw, per in ((dict(), 2), (dict(path=Q.PATH_FUSED), 2), (dict(tile_v=2), 0), (dict(path=Q.PATH_SPLIT), 0),
                        (dict(path=Q.PATH_PLAIN), 0)):
            S.reset()
            r = a.run(itermax=6, **kw)
            assert r["reserved"] == per and (S.launches("k_sor_march") > 0) == (per == 2), kw
        for kw, per in ((dict(), 2), (dict(tile_k=2), 0), (dict(path=Q.PATH_SPLIT), 0)):
            for g in (False, True):
                res, _ = Q.run_batch([a, b], itermax=6, check_every=6, use_graph=g, **kw)
                assert [r["reserved"] for r in res] == [per] * 2, kw
    S.reset()
    with flat_city(Q, 60, 30, 20) as c:
        c.run(itermax=2, path=Q.PATH_SPLIT)
        S.fail_at(1)
        assert c.run(itermax=6)["reserved"] == 0


def case_copies_of_memory_the_runtime_knows(Q, S):
    """Pinned (or device) memory of the caller's is copied by the runtime, not
    through the library's slots, whichever of a call's arrays it is."""
    S.lib.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    with flat_city(Q, 200, 200, 60) as c:
        c.run(itermax=2)
        n = c.city.nface
        for _ in range(4):
            c.get_velocity()  # makes the slots

        def take(pinned):
            out = [np.full(n, 7.0, np.float32) for _ in range(3)]
            for q in pinned:
                p = C.c_void_p()
                assert S.lib.hipHostMalloc(C.byref(p), 4 * n, 0) == 0
                out[q] = np.ctypeslib.as_array((C.c_float * n).from_address(p.value))
                out[q][:] = 7.0
            before = S.value("copied")
            args = [C.cast(a.ctypes.data, C.POINTER(C.c_float)) for a in out]
            assert Q.lib().qesmc_get_velocity(c._h, *args) == Q.OK
            assert not any(a.any() for a in out)
            return S.value("copied") - before

        assert take((0, 1, 2)) == 3
        assert take(()) > 12
        assert 13 < take((1,))


def case_small_members_fill_the_chip(Q, S):
    """Work-groups go to the XCDs in turn: members of a few tiles follow each
    other without gaps (padded to whole eighths, all went to one XCD)."""
    ctxs = [flat_city(Q, 10, 10, 10) for _ in range(32)]
    Q.run_batch(ctxs, itermax=16, check_every=16)
    assert 32 <= S.grid("k_sor_march") < 8 * 32
    for c in ctxs:
        c.close()


def case_batch_beyond_the_cache_is_taken_in_groups(Q, S):
    """Each group has its own launches: two of two iterations, and the one that
    redoes an end inside a launch."""
    from test_gpu_batch_groups import GROUPS, SIZES

    ctxs = [flat_city(Q, *s) for s in SIZES]
    Q.run_batch(ctxs, itermax=4, check_every=4)
    assert S.launches("k_sor_march") == 3 * GROUPS
    for c in ctxs:
        c.close()


def case_batch_replay_of_colour_passes(Q, S):
    """use_graph replays the colour passes of a batch of wall-mask problems."""
    ctxs = [flat_city(Q, 40 + q, 30, 20) for q in range(3)]
    Q.run_batch(ctxs, itermax=8, check_every=8, use_graph=True, path=Q.PATH_SPLIT)
    assert S.value("graph_launches") == 1 and S.launches("k_sor_batch") == 0
    Q.run_batch(ctxs, itermax=8, check_every=8, use_graph=True)
    assert S.value("graph_launches") == 1 and S.launches("k_sor_march") > 0
    for c in ctxs:
        c.close()


def case_thin_towers_take_the_colour_passes(Q, S):
    for dims, march in (((12, 12, 1000), True), ((12, 12, 1300), False), ((20, 20, 1900), True), ((20, 20, 2100), False),
                        ((60, 30, 2500), True), ((100, 30, 2500), True)):
        with flat_city(Q, *dims) as c:
            assert c.run(itermax=4)["reserved"] == (2 if march else 0), dims
            assert c.run(itermax=4, path=Q.PATH_FUSED)["reserved"] == 2


def case_convolutions_at_31_bits(Q, S):
    """A brick's last voxel lies up to 17 voxels beyond six planes: with 48
    channels that passes 31 bits at 1864134 x 2 voxels, whose six planes
    (2147482368 bytes) do not, and there the offsets have 64."""
    for dx, wide in ((1864134, 1), (1864128, 0)):
        S.reset()
        net = Q.UNet(dx, 2, 6, levels=2, base_channels=16, seed=1)
        net.forward(np.zeros((6, 2, dx, 8), np.float32))
        assert S.launches("k_conv_chunksILi16ELb1E") == wide, (dx, S.launches("k_conv_chunks"))
        net.close()


def case_slots_are_made_once_they_repay(Q, S):
    """A context that copies little and goes is not worth the pinned slots; one
    that copies on, or much, makes them, and the last to go frees them."""
    slots = 12

    def held():
        return S.value("host_live")

    for _ in range(8):  # 13 MB each, one context after another
        with flat_city(Q, 128, 128, 64) as c:
            before = held()
            c.get_velocity()
            assert held() == before
    with flat_city(Q, 128, 128, 64) as c:
        before = held()
        made = []
        for _ in range(8):
            c.get_velocity()
            made.append((held() - before) // (4 << 20))
        assert made[0] == 0 and made[-1] == slots and sorted(made) == made, made
        with flat_city(Q, 40, 30, 20):
            pass
        assert held() - before == slots * (4 << 20)
    assert held() < 4 << 20
    with flat_city(Q, 300, 300, 80) as c:  # 90 MB at once
        before = held()
        c.get_velocity()
        assert held() - before == slots * (4 << 20)


CASES = sorted(n for n in globals() if n.startswith("case_"))


@pytest.fixture(scope="session")
def stand_in(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stand_in") / "libamdhip64.so.7")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fPIC", "-shared", "-Wl,-soname,libamdhip64.so.7",
                    os.path.join(ROOT, "tests", "cpp", "hip_stand_in.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("case", CASES)
def test_host_run(stand_in, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case, stand_in], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:] + r.stderr[-4000:])


if __name__ == "__main__":
    S = StandIn(sys.argv[2])
    sys.path.insert(0, os.path.join(ROOT, "qes-public_amd"))
    import qesmc as Q

    globals()[sys.argv[1]](Q, S)
