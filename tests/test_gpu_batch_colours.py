"""Batches of wall-mask problems on the colour passes (path SPLIT): one and two
half-cells per lane, launched directly and replayed, against each member's own
run, bit for bit, warm start and early stops included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(40, 31, 12), (5, 4, 3), (64, 70, 20), (131, 18, 33), (3, 3, 3)]


@pytest.mark.parametrize("tile_v", [1, 2])
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("itermax,tol,every,extend", [(70, -1.0, 32, 0.0), (300, 2e-3, 8, 0.0), (300, 1e-2, 16, 0.25)])
def test_members_match_their_own_runs(qesmc, tile_v, graph, itermax, tol, every, extend):
    kw = dict(itermax=itermax, tol=tol, check_every=every, stop_extend=extend, path=qesmc.PATH_SPLIT)
    ctxs = [qesmc.Context(0) for _ in SIZES]
    try:
        want = []
        for q, (c, (ncx, ncy, ncz)) in enumerate(zip(ctxs, SIZES)):
            blds = qesmc.random_buildings(q, ncx, ncy, 2.0, 4, 6.0, 16.0, 3.0, 8.0, margin=2) if min(ncx, ncy) >= 18 else []
            c.set_city(ncx, ncy, 2.0, qesmc.dz_uniform(ncz, 1.0), blds, (1, 4.0, 10.0, 0.5, 230.0 + 9 * q))
            runs = []
            for _ in range(2):  # the second from the first's lambda
                r = c.run(**kw)
                runs.append((r["iterations"], r["final_max_dlambda"], c.get_lambda()) + tuple(c.get_velocity()))
            want.append(runs)
            c.set_lambda(None)
        for again in range(2):
            res, _ = qesmc.run_batch(ctxs, use_graph=graph, tile_v=tile_v, **kw)
            for q, (c, r) in enumerate(zip(ctxs, res)):
                w = want[q][again]
                assert r["reserved"] == 0 and r["compressed"] == 1 and r["tile_v"] == tile_v
                assert (r["iterations"], r["final_max_dlambda"]) == w[:2], (q, again)
                for a, b in zip((c.get_lambda(),) + tuple(c.get_velocity()), w[2:]):
                    assert np.array_equal(a, b), (q, again)
    finally:
        for c in ctxs:
            c.close()
