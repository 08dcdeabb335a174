"""Solves whose coarsest level has an odd number of cells along x: its red and
black nodes alternate with the row, in one wave, in the whole block with one
and with three nodes of a colour per thread, below strips and in the generic
single-workgroup kernel.  FP64 is the oracle bit for bit, the mixed form
converges."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu

GRIDS = [(104, 64, 4, 1.0, 0), (52, 36, 3, 1.25, 0), (416, 512, 6, 1.0, 0), (208, 32, 5, 1.0, 0),
         (208, 32, 5, 0.8, 10000), (74, 58, 2, 1.0, 0), (122, 114, 2, 1.0, 20000)]


def problem(n1, n2, aspect):
    dom = S.box_domain(n1, n2, Bmode=None)
    rng = np.random.default_rng(n1 + n2)
    phi = np.where(dom.bcnd >= 1, rng.uniform(-5.0, 5.0, dom.bcnd.shape), 0.0)
    inner = dom.bcnd[1:n2 + 2, 1:n1 + 2] == -1
    return dom, (dom.h1, dom.h2 * aspect), phi, np.where(inner, rng.normal(0, 1e-3, inner.shape), 0.0)


@pytest.mark.parametrize("n1,n2,ng,aspect,tail", GRIDS + [(5, 3, 1, 1.0, 0), (37, 29, 1, 1.0, 0), (61, 57, 1, 1.2, 0)])
def test_fp64_matches_oracle(n1, n2, ng, aspect, tail):
    dom, h, phi, b = problem(n1, n2, aspect)
    eps = 1e-5 if ng == 1 else 1e-10
    with L.Context(n1, n2, h[0], h[1], dom.dt, [L.Species(-L.QE, L.ME, 1.0, 16)], ng=ng, mg_tail_nodes=tail) as ctx:
        ctx.set_boundary(dom.bcnd, phi)
        ctx.set_grid(L.GRID_RHS, b)
        info = ctx.iterative_solver(eps=eps, ncycl=200, start=L.START_PREV)
        got = ctx.get_grid(L.GRID_PHI)
    ref = O.iterative_solver(phi, b, dom.bcnd, h, n1, n2, ng, eps=eps)
    assert info["status"] == 0 and info["vcycles"] == ref["vcycles"]
    assert np.array_equal(info["sweeps"], ref["sweeps"][:len(info["sweeps"])])
    assert np.array_equal(got[1:-1, 1:-1], ref["phi"][1:-1, 1:-1])


@pytest.mark.parametrize("n1,n2,ng,aspect,tail", GRIDS)
def test_mixed_converges(n1, n2, ng, aspect, tail):
    dom, h, phi, b = problem(n1, n2, aspect)
    with L.Context(n1, n2, h[0], h[1], dom.dt, [L.Species(-L.QE, L.ME, 1.0, 16)], ng=ng, precision=L.MIXED,
                   mg_tail_nodes=tail) as ctx:
        ctx.set_boundary(dom.bcnd, phi)
        ctx.set_grid(L.GRID_RHS, b)
        info = ctx.iterative_solver(eps=1e-10, ncycl=200, start=L.START_PREV)
        u = ctx.get_grid(L.GRID_PHI)
    assert info["status"] == 0
    aw, an = O.EPS0 / h[0] ** 2, O.EPS0 / h[1] ** 2
    r = b - (aw * (u[1:-1, :-2] + u[1:-1, 2:]) + an * (u[2:, 1:-1] + u[:-2, 1:-1]) - 2.0 * (aw + an) * u[1:-1, 1:-1])
    assert np.abs(r[dom.bcnd[1:-1, 1:-1] == -1]).sum() <= 1.001e-10 * O.mg_alpha(n1, n2, h)
