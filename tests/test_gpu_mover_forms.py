"""The movers' forms by the size of a launch and the cells of a segment: a species
pushed whole takes one of them, its halves (cut between segments) another, and
particles, tallies and densities agree bit for bit."""
import numpy as np
import pytest

import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


def push(dom, E, parts, precision, pushes):
    with L.Context(dom.n1, dom.n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0, len(parts))], zmax=dom.zmax,
                   ngrid=dom.ngrid, precision=precision) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((dom.n2 + 3, dom.n1 + 3)))
        ctx.set_bfield(dom.Bi, dom.nB, dom.hB)
        ctx.set_grid(L.GRID_E, E)
        ctx.upload(1, parts)
        for _ in range(pushes):
            ctx.part_mover(1)
        return ctx.download(1), ctx.get_grid(L.GRID_NP, 1), ctx.mover_tally(1)["p_mac"][0]


# segments of the whole species: mixed above 512 through flat loads (more than 25
# cells a segment) and separate ones, its halves below; FP64 above and below 1024
@pytest.mark.parametrize("precision,n1,n2,segs", [(L.MIXED, 200, 100, 602), (L.MIXED, 110, 100, 602),
                                                  (L.FP64, 200, 100, 1100), (L.FP64, 64, 50, 1026)])
@pytest.mark.parametrize("Bmode,order", [("map", "sorted"), ("coarse", "random"), ("const", "sorted")])
def test_forms_agree(precision, n1, n2, segs, Bmode, order):
    dom = S.box_domain(n1, n2, Bmode=Bmode)
    E = S.random_E(dom, 3e4, seed=2)
    parts = S.particles(dom, segs * 1024 - 300, 1.0e6, seed=n1, edge_frac=0.02)
    if order == "sorted":
        parts = parts[np.lexsort((np.floor(parts[:, 0] / dom.h1), np.floor(parts[:, 1] / dom.h2)))]
    cut = segs // 2 * 1024
    whole, np_w, lost_w = push(dom, E, parts, precision, 2)
    a, np_a, lost_a = push(dom, E, parts[:cut], precision, 2)
    b, np_b, lost_b = push(dom, E, parts[cut:], precision, 2)
    assert np.array_equal(whole, np.concatenate([a, b]))
    assert np.array_equal(lost_w, lost_a + lost_b)
    # whole numbers of 2^-42 or 2^-20 of a particle, scaled and rounded once each
    assert np.abs(np_w - (np_a + np_b)).max() <= 3 * 2.0 ** -53 * np_w.max()


@pytest.mark.parametrize("precision", [L.FP64, L.MIXED])
def test_deposition_forms_agree(precision):
    """513 segments deposit through one window each, their halves through two."""
    dom = S.box_domain(40, 30, Bmode=None)
    parts = S.particles(dom, 513 * 1024 - 5, 1.0, seed=1, edge_frac=0.0)
    parts = parts[np.lexsort((np.floor(parts[:, 0] / dom.h1), np.floor(parts[:, 1] / dom.h2)))]
    out = []
    for sel in (slice(None), slice(0, 256 * 1024), slice(256 * 1024, None)):
        with L.Context(40, 30, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0, len(parts))], zmax=dom.zmax,
                       ngrid=dom.ngrid, precision=precision) as ctx:
            ctx.set_boundary(dom.bcnd, np.zeros((33, 43)))
            ctx.upload(1, parts[sel])
            ctx.charge_deposition(1)
            out.append(ctx.get_grid(L.GRID_NP, 1))
    assert np.abs(out[0] - (out[1] + out[2])).max() <= 3 * 2.0 ** -53 * out[0].max()
