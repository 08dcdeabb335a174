"""Depositions after a call that ended in an error: a failed lepic_create leaves
the runtime's error code to the thread's next call, whose own error return must
not reach the densities, particles and tallies of the calls after it."""
import numpy as np
import pytest

import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu

N1, N2 = 40, 24


def leave_an_error():
    with pytest.raises(L.LepicError):        # 1.6 TB of particles
        L.Context(N1, N2, 1e-4, 1e-4, 1e-12, [L.Species(-L.QE, L.ME, 1.0, 1 << 34)])


def state(ctx):
    return ([ctx.download(p) for p in (1, 2)] + [ctx.get_grid(L.GRID_NP, p) for p in (1, 2)] +
            [ctx.mover_tally(p)["p_mac"][0] for p in (1, 2)])


@pytest.mark.parametrize("precision", [L.FP64, L.MIXED])
@pytest.mark.parametrize("call", ["deposition", "push", "step"])
def test_densities_after_an_error(call, precision):
    dom = S.box_domain(N1, N2, Bmode=None)
    runs = []
    for fail in (False, True):
        with L.Context(N1, N2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0e3, 20_000),
                                                        L.Species(L.QE, 1836 * L.ME, 1.0e3, 20_000)],
                       precision=precision, ng=3) as ctx:
            ctx.set_boundary(dom.bcnd, np.zeros((N2 + 3, N1 + 3)))
            for p in (1, 2):
                ctx.upload(p, S.particles(dom, 15_000, 1.0e6 if p == 1 else 2.0e4, seed=p))
            do = {"deposition": lambda it: [ctx.charge_deposition(p) for p in (1, 2)],
                  "push": lambda it: [ctx.part_mover(p) for p in (1, 2)],
                  "step": lambda it: ctx.step(it, mcc_mode=-1)}[call]
            for p in (1, 2):
                ctx.charge_deposition(p)
            for it in (1, 2):
                do(it)
            before = state(ctx)
            if fail:
                leave_an_error()
                with pytest.raises(L.LepicError):
                    do(3)
                for a, b in zip(state(ctx), before):      # reported before any work
                    assert np.array_equal(a, b)
            do(3)
            after = state(ctx)
            do(4)
            runs.append(after + state(ctx))
    for a, b in zip(*runs):
        assert np.array_equal(a, b)
