"""Network calls on pinned host batches that end in an error: the copies of the
batch are over when the call returns, so its arrays may be overwritten at once,
and the next call on other data is unharmed."""
import os
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "oracle"))
import unet_oracle as U  # noqa: E402
from test_gpu_unet import box_ctx, rand_batch  # noqa: E402

L = pytest.importorskip("jd_lepic_amd")
pytestmark = pytest.mark.gpu


def leave_an_error():
    with pytest.raises(L.LepicError):        # 1.6 TB of particles
        L.Context(16, 16, 1e-4, 1e-4, 1e-12, [L.Species(-L.QE, L.ME, 1.0, 1 << 34)])


@pytest.mark.parametrize("what", ["left error", "empty mask"])
def test_batch_after_an_error(what):
    x, t, m = rand_batch(4, 256, 264, 3)
    pinned = [torch.zeros(a.shape, dtype=torch.float32, pin_memory=True).numpy() for a in (x, t, m)]
    ctx, _ = box_ctx(16)
    with ctx:
        ctx.net_create(capacity=0, seed=1)
        ctx.net_set_params(U.init_params(13))
        loss, g = ctx.net_loss_grad(x, t, m, U.n_params())
        y = ctx.net_forward(x)
        for call in ("grad", "forward"):
            for p, a in zip(pinned, (x, t, m)):
                p[...] = a
            if what == "left error":
                leave_an_error()
            elif call == "forward":
                continue
            else:
                pinned[2][...] = 0.0
            with pytest.raises(L.LepicError):
                if call == "grad":
                    ctx.net_loss_grad(*pinned, U.n_params())
                else:
                    ctx.net_forward(pinned[0])
            for p in pinned:
                p[...] = np.nan
        loss2, g2 = ctx.net_loss_grad(x, t, m, U.n_params())
        y2 = ctx.net_forward(x)
    # FP64 and FP32 sums of atomics in another order
    assert abs(loss2 - loss) <= 1e-12 * loss
    assert np.linalg.norm(g2 - g) <= 1e-5 * np.linalg.norm(g)
    assert np.array_equal(y2, y)
