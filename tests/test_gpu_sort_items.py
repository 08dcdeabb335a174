"""The run sort's forms of 4, 16 and 64 keys per thread on either side of their
switch: the number of runs (2^20 and 2^22, and as few as one block has), with
7-bit and 11-bit digits, where the histogram has room for the form (several
particles of a cell in a segment, so fewer runs than slots)."""
import numpy as np
import pytest

import oracle as O
import scenarios as S

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


def runs_of(cell):
    seg = np.arange(cell.size) // 1024
    return np.unique(seg.astype(np.int64) << 32 | cell).size


# form: keys per thread that the number of runs and the histogram select
@pytest.mark.parametrize("n1,n2,groups,per,form", [
    (128, 128, 1_044_000, 3, 4), (128, 128, 1_050_000, 3, 16), (128, 128, 1_000, 3, 4), (1024, 2048, 200_000, 6, 16),
    (1024, 2048, 200_000, 2, 64)])
def test_sort_forms_match_oracle(n1, n2, groups, per, form):
    count = groups * per
    rng = np.random.default_rng(groups)
    # groups of one cell each; no cell twice in a segment but for its group
    c = rng.permutation(n1 * n2)[np.arange(groups) % (n1 * n2)].repeat(per)
    buckets = 256 if n1 * n2 <= 1 << 16 else 2048
    M, words = runs_of(c), 2048 * (-(-count // 16384))
    fits = {it: -(-M // (256 * it)) * buckets <= words for it in (4, 16)}
    picked = 64 if M > 1 << 22 or not fits[16] else 4 if buckets == 256 and M <= 1 << 20 and fits[4] else 16
    assert picked == form
    dom = S.box_domain(n1, n2, Bmode=None)
    parts = np.zeros((count, 6))
    parts[:, 0] = (c % n1 + rng.uniform(0.1, 0.9, count)) * dom.h1
    parts[:, 1] = (c // n1 + rng.uniform(0.1, 0.9, count)) * dom.h2
    parts[:, 3] = np.arange(count)           # exact in FP32 as well
    with L.Context(n1, n2, dom.h1, dom.h2, dom.dt, [L.Species(-L.QE, L.ME, 1.0, count)], zmax=dom.zmax,
                   ngrid=dom.ngrid, precision=L.MIXED) as ctx:
        ctx.set_boundary(dom.bcnd, np.zeros((n2 + 3, n1 + 3)))
        ctx.upload(1, parts)
        before = ctx.download(1)
        pl = ctx.part_sorting(1, want_plist=True)
        got = ctx.download(1)
    ref, pref = O.part_sorting(n1, n2, (dom.h1, dom.h2), before)
    assert np.array_equal(got, ref) and np.array_equal(pl, pref)
