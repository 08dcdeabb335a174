"""Averaged moments where a particle's place in its coarse cell shows: particles
on the coarse columns, whose cell decides which fine node's factor kq counts,
and columns far from the origin, where an inexact division by the cell's side
would lose digits of the weights.  The weights are the oracle's bit for bit, so
a sum of N terms differs by its order and the terms' products only: (2 N + 8)
2^-53 of the terms' size, four times that in a temperature."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


def both(dom, parts, size_na):
    Nm = 1234.5
    with L.Context(dom.n1, dom.n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, Nm, len(parts))],
                   ngrid=2, track_z=0) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros(dom.bcnd.shape))
        ctx.upload(1, parts)
        ctx.charge_deposition(1)
        dens = ctx.get_grid(L.GRID_NP, 1)
        ctx.moments_accumulate(size_na)
        got, _, _ = ctx.moments()
    pm = O.part_moments(dom, Nm, parts, size_na)
    zero = np.zeros_like(dens)
    return got[0], O.calc_avg(dom, [L.ME], [Nm], [dens], [pm], [zero], size_na, None, srcs=[zero])[0]


@pytest.mark.parametrize("size_na", [1, 2, 4])
def test_particles_on_coarse_columns_and_rows(size_na):
    dom = S.box_domain(512, 256, Bmode=None, ngrid=2)
    # walls on every other fine column and row: kq alternates
    dom.bcnd[3:-3:2, 2:-2] = 2
    dom.bcnd[2:-2, 3:-3:2] = 2
    ha1, ha2 = size_na * dom.h1, size_na * dom.h2
    k, j = np.arange(1, 512 // size_na), np.arange(1, 256 // size_na)
    parts = np.zeros((k.size + j.size, 6))
    parts[:k.size, 0], parts[:k.size, 1] = k * ha1, 3.5 * ha2
    parts[k.size:, 0], parts[k.size:, 1] = 7.5 * ha1, j * ha2
    parts[:, 5] = 1.0e6                       # along z: no half step back
    got, want = both(dom, parts, size_na)
    for q in (0, 4):
        # at most four particles around a node
        assert np.abs(got[..., q] - want[..., q]).max() <= 16 * 2.0 ** -53 * np.abs(want[..., q]).max(), q


@pytest.mark.parametrize("size_na", [1, 2])
def test_temperature_far_from_the_origin(size_na):
    dom = S.box_domain(1024, 1000, Bmode=None)
    rng = np.random.default_rng(size_na)
    n = 6000
    parts = np.zeros((n, 6))
    parts[:, 0] = rng.uniform(960.0, 1020.0, n) * dom.h1
    parts[:, 1] = rng.uniform(940.0, 996.0, n) * dom.h2
    parts[:, 3:] = rng.normal(0.0, 1.0e6, (n, 3))
    got, want = both(dom, parts, size_na)
    ix, iy = (np.floor(parts[:, d] / (size_na * h)).astype(int) for d, h in ((0, dom.h1), (1, dom.h2)))
    per_cell = np.bincount(iy * 2000 + ix).max()
    tol = 4 * (2 * 4 * per_cell + 8) * 2.0 ** -53
    dense = want[..., 0] > 0.1 * want[..., 0].max()
    T, Tw = got[..., 1][dense], want[..., 1][dense]
    assert np.abs(T - Tw).max() <= tol * np.abs(Tw).max()
