"""GPU test of the weight gradient where its split of the image can go wrong:
rows just under, at and over one strip of 128 columns, several strips with a
ragged last one, row ranges that do not divide the height, several images."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "oracle"))
import unet_oracle as U  # noqa: E402
from test_gpu_unet import box_ctx, rand_batch  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,W", [(1, 8, 120), (1, 16, 128), (3, 8, 136), (2, 40, 264), (1, 264, 8), (1, 8, 392)])
def test_weight_gradient_strips(B, H, W):
    ctx, _ = box_ctx(16)
    with ctx:
        ctx.net_create(capacity=0, seed=1)
        flat = U.init_params(13)
        ctx.net_set_params(flat)
        x, t, m = rand_batch(B, H, W, 17)
        _, g = ctx.net_loss_grad(x, t, m, U.n_params())
    _, ref, _ = U.loss_and_grad(x, t, m, flat)
    # Stored tensors are BF16 (half a step is 2^-9): sums in another order
    # flip some of them by a step, through at most 28 of them in a row, so
    # sqrt(28) 2^-9 = 1 % of a layer's gradient in the middle and a few times
    # that for the smallest one.  A row of 8 or a strip's edge column left
    # out (or counted twice) moves the gradient by sqrt(1/W) to sqrt(1/H):
    # 5 % at the widest image.
    o = 0
    for name, ci, co in U.CONV_LAYERS:
        k = 9 * ci * co
        gl, rl = g[o:o + k], ref[o:o + k]
        assert np.linalg.norm(gl - rl) <= 0.05 * np.linalg.norm(rl) + 1e-12, name
        o += k
