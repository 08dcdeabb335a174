"""The payload scatter's order of segments: one by one below four segments
per stripe of an eighth of a row, in stripes from there on, ragged stripes,
a last segment that ends early; every particle at its place either way."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,z", [(L.FP64, 1), (L.MIXED, 1), (L.MIXED, 0)])
@pytest.mark.parametrize("n1,n2,count", [
    (37, 5, 32 * 5 * 1024 - 1024), (37, 5, 32 * 5 * 1024 - 1023), (20, 9, 45 * 9 * 1024 + 7), (6, 3, 150_000), (9, 7, 3)])
def test_sort_in_stripes_matches_oracle(n1, n2, count, precision, z):
    dom = S.box_domain(n1, n2, Bmode=None)
    parts = S.particles(dom, count, 1.0, seed=n1 + count % 1024, edge_frac=0.0)
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0, count)], zmax=dom.zmax,
                   ngrid=dom.ngrid, precision=precision, track_z=z) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((n2 + 3, n1 + 3)))
        ctx.upload(1, parts)
        before = ctx.download(1)
        pl = ctx.part_sorting(1, want_plist=True)
        got = ctx.download(1)
    ref, pref = O.part_sorting(n1, n2, (dom.h1, dom.h2), before)
    assert np.array_equal(got, ref) and np.array_equal(pl, pref)


@pytest.mark.parametrize("n1,n2,count", [(128, 128, 1_000_000), (128, 128, 1_200_000), (128, 128, 4_600_000),
                                         (500, 400, 700_000)])
def test_sort_of_many_runs_matches_oracle(n1, n2, count):
    """Particles in no order, so nearly every one is a run: 4, 16 and 64 keys
    per thread of the run sort (thresholds at 2^20 and 2^22 runs), and 9-bit
    digits."""
    dom = S.box_domain(n1, n2, Bmode=None)
    parts = S.particles(dom, count, 1.0, seed=5, edge_frac=0.0)
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0, count)], zmax=dom.zmax,
                   ngrid=dom.ngrid, precision=L.MIXED) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((n2 + 3, n1 + 3)))
        ctx.upload(1, parts)
        before = ctx.download(1)
        pl = ctx.part_sorting(1, want_plist=True)
        got = ctx.download(1)
    ref, pref = O.part_sorting(n1, n2, (dom.h1, dom.h2), before)
    assert np.array_equal(got, ref) and np.array_equal(pl, pref)
