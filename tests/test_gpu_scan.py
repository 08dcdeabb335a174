"""Exclusive scans of the cell sort and the loader at the edges of a tile (4096
words), of the tiles that a block sums by itself (1024) and on words that no
vector load may take."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2", [(64, 64), (4097, 1 + 3), (67, 63), (2049, 2050)])
def test_load_fills_every_cell(n1, n2):
    dom = S.box_domain(n1, n2, Bmode=None)
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0, 2 * n1 * n2)], zmax=dom.zmax,
                   ngrid=dom.ngrid) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((n2 + 3, n1 + 3)))
        ctx.load_uniform(1, 2, 1.0e5, 0.0, n1 * dom.h1, 7)
        got = ctx.download(1)
    cell = np.floor(got[:, 1] / dom.h2).astype(int) * n1 + np.floor(got[:, 0] / dom.h1).astype(int)
    # cells with four wall corners hold none, the others two, in cell order
    b = dom.bcnd[1:n2 + 2, 1:n1 + 2] >= 1
    open_ = ~(b[:-1, :-1] & b[:-1, 1:] & b[1:, :-1] & b[1:, 1:])
    assert np.array_equal(cell, np.repeat(np.flatnonzero(open_.ravel()), 2))


@pytest.mark.parametrize("count", [4095, 4096, 4097, 70_000])
def test_sort_with_a_run_per_particle(count):
    n1 = n2 = 300
    dom = S.box_domain(n1, n2, Bmode=None)
    parts = S.particles(dom, count, 1.0, seed=count, edge_frac=0.0)
    c = np.random.default_rng(count).permutation(n1 * n2)[:count]
    parts[:, 0], parts[:, 1] = (c % n1 + 0.5) * dom.h1, (c // n1 + 0.5) * dom.h2
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0, count)], zmax=dom.zmax,
                   ngrid=dom.ngrid) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((n2 + 3, n1 + 3)))
        ctx.upload(1, parts)
        pl = ctx.part_sorting(1, want_plist=True)
        got = ctx.download(1)
    ref, pref = O.part_sorting(n1, n2, (dom.h1, dom.h2), parts)
    assert np.array_equal(got, ref) and np.array_equal(pl, pref)
