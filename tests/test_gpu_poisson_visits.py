"""FP64 solves whose multi-block levels exercise every shape of the visit
kernel: launches of 8, 12 and 16 waves, more blocks than CUs, tiles cut by the
grid on both sides, odd sides (ng = 1), cells that are not square, outer walls
that differ from node to node, and a second solve from other wall values; and
levels below them on strips (lanes filled unevenly, one strip per wave) or, too
wide or too many for LDS, in the generic single-workgroup kernel."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


# the 12-wave shapes begin above 256 blocks of 8 waves, the 16-wave ones above
# 256 of 12: 1280 x 768 nodes launch 8, 12 and 16 waves on its levels
@pytest.mark.parametrize("n1,n2,ng,aspect,tail,eps", [
    (101, 67, 1, 1.0, 100, 1e-4), (66, 131, 1, 1.3, 100, 1e-4), (96, 160, 4, 0.7, 100, 1e-10),
    (320, 64, 4, 1.0, 100, 1e-10), (256, 128, 7, 1.0, 0, 1e-10), (160, 160, 5, 0.8, 0, 1e-10),
    (224, 32, 4, 1.0, 0, 1e-10), (512, 32, 5, 1.0, 0, 1e-10), (192, 192, 6, 1.0, 10000, 1e-10), (1280, 768, 8, 1.0, 0, 1e-7), (1280, 768, 8, 1.2, 2000, 1e-7)])
def test_fp64_visits_match_oracle(n1, n2, ng, aspect, tail, eps):
    dom = S.box_domain(n1, n2, Bmode=None)
    h = (dom.h1, dom.h2 * aspect)
    bc = dom.bcnd.copy()
    a1, a2 = n1 // 4 // 8 * 8 + 1, n2 // 4 // 8 * 8 + 1
    bc[a2:a2 + n2 // 8 // 8 * 8 + 1, a1:a1 + n1 // 8 // 8 * 8 + 1] = 2
    rng = np.random.default_rng(n1 + 3 * n2)
    wall = bc >= 1
    phi = np.where(wall, rng.uniform(-5.0, 5.0, bc.shape), 0.0)
    inner = bc[1:n2 + 2, 1:n1 + 2] == -1
    with L.Context(n1, n2, h[0], h[1], dom.dt, [L.Species(-L.QE, L.ME, 1.0, 16)], ng=ng, ngrid=2,
                   mg_tail_nodes=tail) as ctx:
        ref_phi = phi
        for turn in range(2):
            if turn:               # other wall values, the nodes between them as they are
                ref_phi = np.where(wall, phi * 1.5, ref_phi)
            ctx.set_boundary(bc, ref_phi)
            b = np.where(inner, rng.normal(0, 1e-3, inner.shape), 0.0)
            ctx.set_grid(L.GRID_RHS, b)
            info = ctx.iterative_solver(eps=eps, start=L.START_PREV)
            got = ctx.get_grid(L.GRID_PHI)
            ref = O.iterative_solver(ref_phi, b, bc, h, n1, n2, ng, eps=eps)
            ref_phi = ref["phi"]
            # a sweep's bits are the oracle's; the L1 sums differ in their
            # order, which the sweep counts do not see unless a ratio of
            # residuals lies within 1e-13 of the exit test's 0.6
            assert info["vcycles"] == ref["vcycles"], turn
            assert np.array_equal(info["sweeps"], ref["sweeps"][:len(info["sweeps"])]), turn
            assert np.array_equal(got[1:-1, 1:-1], ref_phi[1:-1, 1:-1]), turn


@pytest.mark.parametrize("precision,n1,n2,ng", [
    (L.FP64, 5, 3, 1), (L.FP64, 7, 12, 1), (L.FP64, 130, 66, 2), (L.FP64, 2050, 6, 2), (L.MIXED, 12, 8, 3),
    (L.MIXED, 48, 264, 4), (L.MIXED, 1600, 1400, 4)])
def test_starting_residual(precision, n1, n2, ng):
    """The finest level's residual where its threads' two columns and four
    rows meet the walls, in one block and in more blocks than it has."""
    dom = S.box_domain(n1, n2, Bmode=None)
    bc = dom.bcnd.copy()
    if n1 > 40:
        bc[4:6, 9:30] = 2
    rng = np.random.default_rng(n1)
    phi = rng.uniform(-5.0, 5.0, bc.shape)
    b = rng.normal(0, 1e-3, (n2 + 1, n1 + 1))
    with L.Context(n1, n2, dom.h1, dom.h2 * 1.25, dom.dt, [L.Species(-L.QE, L.ME, 1.0, 16)], ng=ng, ngrid=2,
                   precision=precision) as ctx:
        ctx.set_boundary(bc, phi)
        ctx.set_grid(L.GRID_RHS, b)
        info = ctx.iterative_solver(eps=1e30, start=L.START_PREV)
    aw, an = O.EPS0 / dom.h1 ** 2, O.EPS0 / (dom.h2 * 1.25) ** 2
    u = phi[1:-1, 1:-1]
    r = b - (aw * (phi[1:-1, :-2] + phi[1:-1, 2:]) + an * (phi[2:, 1:-1] + phi[:-2, 1:-1]) - 2.0 * (aw + an) * u)
    ref = np.abs(r[bc[1:-1, 1:-1] == -1]).sum() / O.mg_alpha(n1, n2, (dom.h1, dom.h2 * 1.25))
    # sums of up to 2.2e6 positive terms in two orders, and terms that cancel
    # to 1e-2 of their parts
    assert abs(info["res0"] - ref) <= 1e-11 * ref
