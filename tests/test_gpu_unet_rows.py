"""A batch with more rows of pixels than a grid has blocks along y (65535), on
the finest level and on the one below: its gradient is the mean of its halves'
(the scale of the loss differs by an exact factor of two, so every stored BF16
value has the same mantissa).  FP32 sums of 1e6 terms of either sign in another
order: sqrt(1e6) 2^-24 = 6e-5 of a layer's norm; rows left out or taken twice
move it by their share, a part in three and more."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "oracle"))
import unet_oracle as U  # noqa: E402
from test_gpu_unet import box_ctx  # noqa: E402

pytestmark = pytest.mark.gpu


def test_gradient_of_many_rows():
    B, H, W = 16400, 8, 8              # 131200 rows, 65600 on the second level
    rng = np.random.default_rng(3)
    x = rng.standard_normal((B, H, W, 2), dtype=np.float32)
    t = rng.standard_normal((B, H, W), dtype=np.float32)
    m = np.ones((B, H, W), np.float32)
    ctx, _ = box_ctx(16)
    with ctx:
        ctx.net_create(capacity=0, seed=1)
        ctx.net_set_params(U.init_params(13))
        loss, g = ctx.net_loss_grad(x, t, m, U.n_params())
        parts = [ctx.net_loss_grad(x[s], t[s], m[s], U.n_params()) for s in (slice(0, B // 2), slice(B // 2, B))]
    assert abs(loss - 0.5 * (parts[0][0] + parts[1][0])) <= 1e-9 * loss
    want = 0.5 * (parts[0][1] + parts[1][1])
    o = 0
    for name, ci, co in U.CONV_LAYERS + [("out", 16, 1)]:
        k = (9 if name != "out" else 1) * ci * co
        assert np.linalg.norm(g[o:o + k] - want[o:o + k]) <= 1e-3 * np.linalg.norm(want[o:o + k]), name
        o += k
