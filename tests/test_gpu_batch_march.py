"""Batches that march (two iterations per launch, every member wall-mask
encoded): the members' results are those of their own runs, bit for bit,
wherever the run ends within a launch, a polling interval or a replay, and
for batches that are taken in groups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL = [(5, 4, 3), (40, 31, 12), (64, 70, 20), (131, 18, 33), (3, 3, 3)]
LARGE = [(210, 200, 170), (20, 20, 10), (260, 180, 160), (190, 210, 170)]  # 285 MB of arrays: groups


def problem(qesmc, oracle, ncx, ncy, ncz, seed):
    blds = qesmc.random_buildings(seed, ncx, ncy, 2.0, 4, 6.0, 16.0, 3.0, 8.0, margin=2) if min(ncx, ncy) >= 18 else []
    return oracle.build_city(ncx, ncy, 2.0, oracle.dz_uniform(ncz, 1.0), blds, (1, 4.0, 10.0, 0.5, 230.0 + 9 * seed))


@pytest.mark.parametrize("sizes,itermax,tol,every,graph,extend", [
    (SMALL, 1, -1.0, 64, False, 0.0), (SMALL, 2, -1.0, 64, True, 0.0), (SMALL, 41, -1.0, 7, False, 0.0),
    (SMALL, 41, -1.0, 7, True, 0.0), (SMALL, 300, 2e-3, 8, False, 0.0), (SMALL, 300, 2e-3, 5, True, 0.0),
    (SMALL, 300, 1e-2, 16, True, 0.25), (LARGE, 13, -1.0, 4, False, 0.0), (LARGE, 60, 3e-2, 5, True, 0.0)])
def test_members_match_their_own_runs(qesmc, oracle, sizes, itermax, tol, every, graph, extend):
    probs = [problem(qesmc, oracle, *s, seed) for seed, s in enumerate(sizes)]
    kw = dict(itermax=itermax, tol=tol, check_every=every, stop_extend=extend)
    want = []
    for p in probs:
        with qesmc.Context(0) as ctx:
            ctx.set_geometry(p)
            ctx.set_inflow(p.u0, p.v0, p.w0)
            r = ctx.run(**kw)
            want.append((r["iterations"], r["final_max_dlambda"], ctx.get_lambda()) + tuple(ctx.get_velocity()))
    ctxs = [qesmc.Context(0) for _ in probs]
    try:
        for ctx, p in zip(ctxs, probs):
            ctx.set_geometry(p)
            ctx.set_inflow(p.u0, p.v0, p.w0)
        for again in range(2):  # a second batch on the same contexts, from lambda = 0
            for ctx in ctxs:
                ctx.set_lambda(None)
            res, _ = qesmc.run_batch(ctxs, use_graph=graph, **kw)
            for i, (r, ctx) in enumerate(zip(res, ctxs)):
                assert (r["iterations"], r["final_max_dlambda"]) == want[i][:2], i
                for a, b in zip((ctx.get_lambda(),) + tuple(ctx.get_velocity()), want[i][2:]):
                    assert np.array_equal(a, b), i
    finally:
        for ctx in ctxs:
            ctx.close()
    if tol > 0 and sizes is SMALL:
        assert len({w[0] for w in want}) > 1 and max(w[0] for w in want) < itermax
