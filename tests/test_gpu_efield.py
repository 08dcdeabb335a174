"""Electric field in one pass: interior, walls and the FP32 copy of a mixed
context, on sides around the blocks' 128 columns, with wall blocks a cell apart
(a wall's extrapolation meets another wall: serial pass) and further."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["FP64", "MIXED"])
@pytest.mark.parametrize("n1,n2,gap", [(12, 8, 0), (125, 9, 3), (126, 10, 2), (140, 24, 3), (140, 24, 2)])
def test_field_and_its_copy(n1, n2, gap, precision):
    dom = S.box_domain(n1, n2, Bmode=None)
    bc = dom.bcnd.copy()
    if gap:
        bc[4:6, 5] = 1
        bc[4:6, 5 + gap] = 1
    rng = np.random.default_rng(n1 + gap)
    phi = rng.normal(0, 10.0, bc.shape)
    E0 = rng.normal(0, 1e3, bc.shape + (2,))
    ref = O.calc_efield(n1, n2, (dom.h1, dom.h2), phi, bc, E0.copy())
    parts = S.particles(dom, 5000, 1.0e6, seed=n2)
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0, 6000)], ngrid=dom.ngrid,
                   precision=getattr(L, precision)) as ctx:
        ctx.set_boundary(bc, np.zeros(bc.shape))
        ctx.set_grid(L.GRID_E, E0)
        ctx.set_grid(L.GRID_PHI, phi)
        ctx.calc_efield()
        E = ctx.get_grid(L.GRID_E)
        ctx.upload(1, parts)
        ctx.part_mover(1)
        got = ctx.download(1)
        # the same push from a field set by the host, which makes the copy itself
        ctx.set_grid(L.GRID_E, E)
        ctx.upload(1, parts)
        ctx.part_mover(1)
        want = ctx.download(1)
    assert np.array_equal(E, ref)
    assert np.array_equal(got, want)
