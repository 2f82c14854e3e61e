"""Marching batches taken in several groups (arrays beyond the Infinity
Cache): every member's result is that of its own run, bit for bit, with ends
inside a launch in every group.  That these sizes make three groups is checked
in test_host_runs.py, whatever walls they hold."""
import numpy as np
import pytest

SIZES = [(220 + q % 3, 200, 60 - q % 2) for q in range(12)]  # 398 MB; the groups are the thirds
GROUPS = 3


@pytest.mark.gpu
@pytest.mark.parametrize("itermax,stop,every,extend", [(13, 0, 4, 0.0), (120, 41, 5, 0.0), (120, 30, 8, 0.3)])
def test_members_of_every_group_match_their_own_runs(qesmc, itermax, stop, every, extend):
    """stop: the tolerance is the largest max|dlambda| of all members after so
    many iterations, by which most have stopped (0: none); the winds are weak
    ones, so that it is below the 1.0 that lets iteration 0 run."""
    ctxs = [qesmc.Context(0) for _ in SIZES]
    try:
        for q, (c, (ncx, ncy, ncz)) in enumerate(zip(ctxs, SIZES)):
            blds = qesmc.random_buildings(70 + q, ncx, ncy, 2.0, 20 + 5 * q, 8.0, 30.0, 4.0, 30.0, margin=2)
            c.set_city(ncx, ncy, 2.0, qesmc.dz_uniform(ncz, 1.0), blds, (1, 0.03 + 0.004 * q, 10.0, 0.5, 230.0 + 9 * q))
        tol = max([c.run(itermax=stop, tol=-1.0)["final_max_dlambda"] for c in ctxs if stop], default=-1.0)
        kw = dict(itermax=itermax, tol=tol, check_every=every, stop_extend=extend)
        want = []
        for c in ctxs:
            c.set_lambda(None)
            r = c.run(**kw)
            want.append((r["iterations"], r["final_max_dlambda"], c.get_lambda()) + tuple(c.get_velocity()))
            c.set_lambda(None)
        res, _ = qesmc.run_batch(ctxs, **kw)
        for q, (c, r) in enumerate(zip(ctxs, res)):
            assert r["reserved"] == 2 and (r["iterations"], r["final_max_dlambda"]) == want[q][:2], q
            for a, b in zip((c.get_lambda(),) + tuple(c.get_velocity()), want[q][2:]):
                assert np.array_equal(a, b), q
    finally:
        for c in ctxs:
            c.close()
    ends = [w[0] for w in want]
    print(ends)
    if tol > 0:
        third = len(SIZES) // GROUPS
        for g in range(GROUPS):  # an end after the first iteration of a launch
            assert any(e % 2 and e < itermax for e in ends[g * third:(g + 1) * third]), ends
