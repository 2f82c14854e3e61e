"""The march (two iterations per launch, QESMC_PATH_AUTO on a wall mask)
against the oracle, bit for bit, where its tiling can go wrong: domains at the
edges of its tiles (32 or 64 half-cells less the halo, 16 to 64 rows), of
one plane and of a segment's halo more or less, odd and even iteration
counts, runs that end inside a launch, walls above open planes, refreshes
at odd intervals, and a run that finds no wall values at all in a layer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

AUTO, SPLIT, FUSED = 0, 2, 3


def same(a, b, what):
    assert a.shape == b.shape and np.array_equal(a, b, equal_nan=True), (what, int((a != b).sum()))


def city(O, Q, ncx, ncy, ncz, seed=5, nb=5):
    dz = Q.dz_geometric(ncz, 1.0, 1.02)
    blds = Q.random_buildings(seed, ncx, ncy, 2.0, nb, 4.0, 20.0, 2.0, 0.4 * float(dz[1:].sum()), margin=1) \
        if min(ncx, ncy) > 14 else []
    return O.build_city(ncx, ncy, 2.0, dz, blds, (1, 4.0, 10.0, 0.5, 213.0))


# (ncx, ncy, ncz): 64 / 65 / 66 cells are 32 / 33 / 33 half-cells (one x tile or two), 120 and 122 the
# second tile's edge; 16, 17, 24, 25, 32, 33 rows the y tiles'; few planes, and one more than a segment
@pytest.mark.parametrize("shape", [(64, 16, 9), (65, 17, 8), (66, 24, 5), (120, 25, 4), (121, 33, 3), (122, 32, 12),
                                   (5, 5, 3), (4, 70, 2), (3, 3, 1), (129, 65, 19), (30, 200, 33), (257, 66, 7)])
@pytest.mark.parametrize("itermax", [1, 2, 9])
def test_tile_edges(gpu_ctx, oracle, qesmc, shape, itermax):
    p = city(oracle, qesmc, *shape)
    rng = np.random.default_rng(3)
    lam0 = rng.normal(0.0, 3.0, p.ncell).astype(np.float32)
    for start in (None, lam0):
        u, v, w, lam, res = gpu_ctx.solve(p, start, itermax=itermax, tol=-1.0, path=AUTO)
        ou, ov, ow, olam, oit, ome = oracle.solve_rb_f32(p, lam=start, itermax=itermax, tol=-1.0)
        assert res["iterations"] == oit == itermax
        assert np.float32(res["final_max_dlambda"]) == np.float32(ome)
        same(lam, olam, "lambda")
        for g, o, n in ((u, ou, "u"), (v, ov, "v"), (w, ow, "w")):
            same(g, o, n)


@pytest.mark.parametrize("tile_k", [1, 4, 5, 30])
def test_segments(gpu_ctx, oracle, qesmc, tile_k):
    p = city(oracle, qesmc, 90, 50, 31)
    lam = gpu_ctx.solve(p, itermax=11, tol=-1.0, path=FUSED, tile_k=tile_k)[3]
    same(lam, oracle.solve_rb_f32(p, itermax=11, tol=-1.0)[3], "lambda")


@pytest.mark.parametrize("check_every", [1, 3, 64])
def test_end_inside_a_launch(gpu_ctx, oracle, qesmc, check_every):
    """A tolerance that the reference's rule meets after an odd and after an
    even number of iterations, with and without the production rule."""
    p = city(oracle, qesmc, 70, 60, 20)
    ends = {}
    for n in range(20, 40):  # max|dlambda| after n iterations, as the tolerance
        tol = float(np.float32(oracle.solve_rb_f32(p, itermax=n, tol=-1.0)[5]))
        it = oracle.solve_rb_f32(p, itermax=400, tol=tol)[4]
        ends.setdefault(it % 2, (it, tol))
        if len(ends) == 2:
            break
    assert len(ends) == 2
    for it, tol in ends.values():
        u, v, w, lam, res = gpu_ctx.solve(p, itermax=400, tol=tol, path=AUTO, check_every=check_every)
        ou, ov, ow, olam, oit, ome = oracle.solve_rb_f32(p, itermax=400, tol=tol)
        assert res["iterations"] == oit == it
        assert np.float32(res["final_max_dlambda"]) == np.float32(ome)
        same(lam, olam, "lambda")
        same(u, ou, "u")
        # a second run goes on from what the first left
        lam2 = gpu_ctx.solve(p, lam, itermax=3, tol=-1.0, path=AUTO)[3]
        same(lam2, oracle.solve_rb_f32(p, lam=olam, itermax=3, tol=-1.0)[3], "lambda, continued")
        for ext in (0.1, 0.5):
            kw = dict(itermax=400, tol=tol, check_every=check_every, stop_extend=ext)
            a = gpu_ctx.solve(p, path=AUTO, **kw)
            b = gpu_ctx.solve(p, path=SPLIT, **kw)
            assert a[4]["iterations"] == b[4]["iterations"]
            same(a[3], b[3], "lambda, production rule")


@pytest.mark.parametrize("every", [1, 3, 4, 7])
@pytest.mark.parametrize("tol", [-1.0, 2e-2])
def test_refreshes(gpu_ctx, oracle, qesmc, every, tol):
    p = city(oracle, qesmc, 75, 41, 18)
    kw = dict(itermax=60, tol=tol, omega=1.93, refine_every=every)
    a = gpu_ctx.solve(p, path=AUTO, **kw)
    b = gpu_ctx.solve(p, path=SPLIT, **kw)
    assert a[4]["iterations"] == b[4]["iterations"]
    assert a[4]["final_max_dlambda"] == b[4]["final_max_dlambda"]
    same(a[3], b[3], "lambda")
    same(a[2], b[2], "w")


def test_walls_above_open_planes(gpu_ctx, oracle, qesmc):
    """A slab hanging over open planes, and a layer where every wall value of
    one direction is gone: still a wall mask."""
    p = city(oracle, qesmc, 80, 48, 40, nb=0)
    k, j, i = 25, slice(10, 30), slice(20, 60)
    shape = (p.nz - 1, p.ny - 1, p.nx - 1)
    for arr, sel in ((p.m, (k, j, i)), (p.n, (k + 1, j, i)), (p.m, (33, slice(None), slice(None))),
                     (p.n, (34, slice(None), slice(None)))):
        arr.reshape(shape)[sel] = 0.0
    for itermax in (8, 9):
        res = gpu_ctx.solve(p, itermax=itermax, tol=-1.0, path=AUTO)
        assert res[4]["compressed"] == 1
        same(res[3], oracle.solve_rb_f32(p, itermax=itermax, tol=-1.0)[3], "lambda")


def test_non_finite_lambda_is_reported(gpu_ctx, oracle, qesmc):
    p = city(oracle, qesmc, 40, 30, 10)
    for bad in (np.float32(np.nan), np.float32(np.inf)):
        lam0 = np.zeros(p.ncell, np.float32)
        lam0.reshape(p.nz - 1, p.ny - 1, p.nx - 1)[5, 12, 17] = bad
        for itermax in (1, 2, 5):
            with pytest.raises(qesmc.QesmcError) as e:
                gpu_ctx.solve(p, lam0, itermax=itermax, tol=-1.0, path=AUTO)
            assert e.value.code == qesmc.ERR_NONFINITE
