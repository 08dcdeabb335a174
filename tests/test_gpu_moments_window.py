"""k_part_moments away from the sorted state it is tuned for: particles in
random order (runs of one particle, most of them outside the segment's LDS
window), a species of one particle, a last segment of a few slots, particles
of one coarse cell only, and particles within a step of the walls; against the
oracle's part_moments.  FP64 sums of at most 1e5 terms in another order:
1e-11 of the largest moment; mixed: the FP32 state's rounding, 2e-5."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(L.FP64, 1e-11), (L.MIXED, 2e-5)])
@pytest.mark.parametrize("count,size_na,order", [(20_000, 1, "random"), (20_003, 2, "sorted"), (1, 1, "random"),
                                                 (1_030, 4, "one cell")])
def test_moments_of_any_order(prec, tol, count, size_na, order):
    n1, n2 = 160, 48
    dom = S.box_domain(n1, n2, Bmode=None)
    parts = S.particles(dom, count, 1.0e6, seed=count, edge_frac=0.1)
    if order == "one cell":
        parts[:, 0] = (81.0 + 0.9 * np.random.default_rng(1).random(count)) * dom.h1
        parts[:, 1] = (21.0 + 0.9 * np.random.default_rng(2).random(count)) * dom.h2
        parts[:, 3:5] *= 1e-3            # half a step stays in the coarse cell
    Nm = 1234.5
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, Nm, count + 16)], precision=prec,
                   track_z=0) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((n2 + 3, n1 + 3)))
        ctx.upload(1, parts)
        if order == "sorted":
            ctx.part_sorting(1)
        ctx.charge_deposition(1)
        held = ctx.download(1)
        dens = ctx.get_grid(L.GRID_NP, 1)
        ctx.moments_accumulate(size_na)
        got, _, _ = ctx.moments()
    pm = O.part_moments(dom, Nm, held, size_na)
    zero = np.zeros_like(dens)
    want = O.calc_avg(dom, [L.ME], [Nm], [dens], [pm], [zero], size_na, None, srcs=[zero])
    for q in (0, 2, 3, 4):               # density and currents
        assert np.abs(got[0, ..., q] - want[0, ..., q]).max() <= tol * np.abs(want[0, ..., q]).max(), q
    # the temperature divides by the density: nodes that hold a tenth of the peak
    dense = want[0, ..., 0] > 0.1 * want[0, ..., 0].max()
    T, Tw = got[0, ..., 1][dense], want[0, ..., 1][dense]
    assert np.abs(T - Tw).max(initial=0.0) <= 100 * tol * np.abs(Tw).max(initial=0.0)
