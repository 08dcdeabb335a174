"""FP64 push through the field tile, bit for bit against the oracle: domains
smaller and larger than the tile (32 x 10 nodes), particles in cell order (all
in the tile) and in none (most outside it), segments that end early."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Bmode", ["map", None])
@pytest.mark.parametrize("n1,n2,count,ordered", [
    (12, 6, 1, True), (12, 6, 1023, False), (31, 9, 1024, True), (33, 11, 1025, True), (90, 50, 20001, True),
    (90, 50, 20001, False)])
def test_fp64_push_through_the_tile(n1, n2, count, ordered, Bmode):
    dom = S.box_domain(n1, n2, Bmode=Bmode, Bpeak=0.05)
    parts = S.particles(dom, count, 1.0e6, seed=n1 + count)
    if ordered:
        parts = parts[np.lexsort(((parts[:, 0] / dom.h1).astype(int), (parts[:, 1] / dom.h2).astype(int)))]
    Ei = S.random_E(dom, 5e4, seed=3)
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 55.0, count + 10)], zmax=dom.zmax,
                   ngrid=dom.ngrid) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((n2 + 3, n1 + 3)))
        if Bmode:
            ctx.set_bfield(dom.Bi, dom.nB, dom.hB)
        ctx.upload(1, parts)
        ctx.set_grid(L.GRID_E, Ei)
        ctx.part_mover(1, deposit=True)
        got, rho = ctx.download(1), ctx.get_grid(L.GRID_NP, 1)
    ref = O.part_mover(dom, -L.QE, L.ME, 55.0, Ei, parts, np.zeros(len(parts), np.int8))
    assert np.array_equal(got, ref["vxp"])
    rho_ref = O.charge_deposition(dom, 55.0, ref["vxp"])
    # a run's weights are rounded to 2^-42 of a particle, the oracle's sums to
    # 2^-53 of a node: under 1e-12 of the fullest node
    assert np.abs(rho - rho_ref).max() <= 1e-12 * max(np.abs(rho_ref).max(), 1e-300)


@pytest.mark.parametrize("z", [0, 1])
def test_mixed_push_is_the_same_in_both_launch_forms(z):
    """512 segments take one form of the kernel, 513 the other: the particles
    they share come out with the same bits."""
    n = 512 * 1024
    dom = S.box_domain(64, 48, Bmode="map", Bpeak=0.05)
    parts = S.particles(dom, n + 1, 1.0e6, seed=8, edge_frac=0.0)
    parts = parts[np.lexsort(((parts[:, 0] / dom.h1).astype(int), (parts[:, 1] / dom.h2).astype(int)))]
    Ei = S.random_E(dom, 5e4, seed=3)
    out = []
    for count in (n, n + 1):
        with L.Context(64, 48, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 55.0, n + 2048)], zmax=dom.zmax,
                       ngrid=dom.ngrid, precision=L.MIXED, track_z=z) as ctx:
            ctx.set_boundary(dom.bcnd, np.zeros((51, 67)))
            ctx.set_bfield(dom.Bi, dom.nB, dom.hB)
            ctx.upload(1, parts[:count])
            ctx.set_grid(L.GRID_E, Ei)
            ctx.part_mover(1, deposit=True)
            out.append(ctx.download(1))
    assert len(out[0]) > 0.9 * n
    assert np.array_equal(out[0], out[1][:len(out[0])])


@pytest.mark.parametrize("precision", [L.FP64, L.MIXED])
@pytest.mark.parametrize("n1,n2,per_cell,push", [(96, 20, 30, True), (96, 20, 30, False), (300, 9, 7, True), (300, 9, 7, False)])
def test_density_of_segments_over_the_end_of_a_row(n1, n2, per_cell, push, precision):
    """Particles in cell order whose segments run over the end of a row of
    cells, and (7 per cell) over 146 columns, more than either window holds."""
    dom = S.box_domain(n1, n2, Bmode=None)
    count = per_cell * n1 * n2
    parts = S.particles(dom, count, 1.0, seed=n1, edge_frac=0.0)
    parts = parts[np.lexsort(((parts[:, 0] / dom.h1).astype(int), (parts[:, 1] / dom.h2).astype(int)))]
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 55.0, count)], zmax=dom.zmax,
                   ngrid=dom.ngrid, precision=precision) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((n2 + 3, n1 + 3)))
        ctx.upload(1, parts)
        if push:
            ctx.part_mover(1, deposit=True)
        else:
            ctx.charge_deposition(1)
        now, rho = ctx.download(1), ctx.get_grid(L.GRID_NP, 1)
    ref = O.charge_deposition(dom, 55.0, now)
    # mixed: every weight is rounded to 2^-20 (half: 4.8e-7) from FP32 factors
    # (2^-23), and four times a cell's particles touch a node; FP64: 2^-42
    tol = 4 * (2.0 ** -21 + 2.0 ** -22) if precision == L.MIXED else 1e-12
    assert np.abs(rho - ref).max() <= tol * np.abs(ref).max()
