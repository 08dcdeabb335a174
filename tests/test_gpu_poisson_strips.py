"""The mixed form's multigrid on register strips: a level's visit gives the
same bits in the tiled kernel (k_tile32), in the single-workgroup kernel
(k_tail_strips) and in the generic single-workgroup kernel, so phi must not depend
on mg_tail_nodes as long as the finest level stays tiled.  Sides whose strips
fill their lanes unevenly, cells that are not square, a grid electrode, and a
level too wide for the strips of k_tail_strips (512 x 32)."""
import numpy as np
import pytest

import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


def solve(n1, n2, ng, tail, aspect):
    dom = S.box_domain(n1, n2, Bmode=None)
    bc = dom.bcnd.copy()
    phi = np.zeros((n2 + 3, n1 + 3))
    phi[n2 + 1:, :] = 10.0
    a1, a2 = n1 // 4 + 1, n2 // 4 + 1          # electrode edges on odd node indices
    bc[a2:a2 + n2 // 8 + 1, a1:a1 + n1 // 8 + 1] = 2
    phi[bc == 2] = 25.0
    b = np.random.default_rng(n1 + n2).normal(0, 1e-3, (n2 + 1, n1 + 1))
    b[bc[1:n2 + 2, 1:n1 + 2] != -1] = 0.0
    out = []
    with L.Context(n1, n2, dom.h1, dom.h2 * aspect, dom.dt, [L.Species(-L.QE, L.ME, 1.0, 16)], ng=ng, ngrid=2,
                   precision=L.MIXED, mg_tail_nodes=tail) as ctx:
        ctx.set_boundary(bc, phi)
        for scale in (1.0, 1.1):
            ctx.set_grid(L.GRID_RHS, b * scale)
            info = ctx.iterative_solver(eps=1e-7, start=L.START_PREV)
            assert info["res"] <= 1e-7 and info["status"] == 0
            out.append(ctx.get_grid(L.GRID_PHI))
    return out


@pytest.mark.parametrize("n1,n2,ng,aspect,tails", [
    (128, 128, 7, 1.0, (0, 400, 100)), (160, 160, 5, 1.0, (0, 200)), (192, 96, 6, 1.25, (0, 100)),
    (272, 80, 4, 0.8, (0, 500)), (512, 32, 5, 1.0, (0, 100)), (1024, 256, 8, 1.0, (0, 20000))])
def test_phi_does_not_depend_on_the_levels_layout(n1, n2, ng, aspect, tails):
    first = solve(n1, n2, ng, tails[0], aspect)
    for tail in tails[1:]:
        for a, b in zip(first, solve(n1, n2, ng, tail, aspect)):
            assert np.array_equal(a, b), tail
