"""The Lanczos step of the over-relaxation estimate on a mask-encoded geometry
(waves of 64 cells marching along k) against the step that reads the
coefficients, at ragged sizes."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncx,ncy,ncz", [(5, 4, 3), (66, 5, 9), (67, 7, 10), (68, 9, 12), (131, 18, 33), (200, 40, 25)])
def test_masked_step_matches_general(qesmc, oracle, ncx, ncy, ncz):
    blds = qesmc.random_buildings(3, ncx, ncy, 2.0, 4, 6.0, 16.0, 3.0, 8.0, margin=2) if ncy >= 18 else []
    p = oracle.build_city(ncx, ncy, 2.0, oracle.dz_uniform(ncz, 1.0), blds, (1, 4.0, 10.0, 0.5, 270.0))
    # a solid cell, whose own coefficients the operator does not use: one that
    # no wall mask encodes leaves the operator as it is and takes the general step
    NX, NY = p.nx - 1, p.ny - 1
    c = 1 + NX + NX * NY
    p.icellflag[c] = 0
    with qesmc.Context(0) as ctx:
        # fewer steps than cells: past that the Krylov space is exhausted, and what
        # follows is rounding
        for steps in (1, 2, 5 if ncx == 5 else 35):
            p.coeffs[0][c] = 1.0 / 4.0
            ctx.set_geometry(p)
            a, oa = ctx.estimate_omega(steps=steps)
            p.coeffs[0][c] = 0.37
            ctx.set_geometry(p)
            b, ob = ctx.estimate_omega(steps=steps)
            # the same products in FP64, summed in another order
            assert 0.0 < b < 1.0
            assert abs(a - b) <= 1e-11
            assert abs(oa - ob) <= 1e-6
