"""The row-block MLP kernels (k_mlp_rows, k_mlp_weights) at the edges of
their tiles: batches around the 4, 8 and 16 rows of a workgroup and the 32
of a weight-gradient step, widths that are no multiple of a 16-column block
or of the 128-wide padding, one layer, and the widest network they take."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as mo  # noqa: E402

from cudaprotoplanetarydisks_amd.mlp import MLP  # noqa: E402

pytestmark = pytest.mark.gpu

CASES = [  # widths, batch
    ([5, 64, 48], 1), ([5, 70, 33, 45], 31), ([3, 16, 17], 33), ([7, 20], 65), ([130, 129, 300, 9], 100),
    ([5, 64, 48], 1029), ([5, 70, 33], 2051), ([5, 896, 7], 20), ([5, 900, 7], 20),
]


@pytest.mark.parametrize("widths, batch", CASES)
def test_gradient_and_step(widths, batch):
    """Gradient against the CPU reference with the same BF16 rounding points
    (the tolerances of tests/test_gpu_mlp.py); then two Adam steps, whose
    first loss is the gradient call's and whose parameters follow from the
    gradients: |step| <= lr (1 + 1e-3) per step, the first one lr * sign(g)
    wherever |g| is far above Adam's 1e-8."""
    rng = np.random.default_rng(batch)
    x = rng.uniform(-1, 1, size=(batch, widths[0])).astype(np.float32)
    t = rng.normal(size=(batch, widths[-1])).astype(np.float32)
    with MLP(widths, max_batch=batch + 3, seed=11) as net:
        p0 = net.params()
        loss, g = net.gradient(x, t)
        losses = net.train(x, t, batch=batch, steps=1, lr=1e-3)
        p1 = net.params()
    ref_loss, ref_g = mo.loss_and_grad(p0, widths, x, t, emulate_bf16=True)
    assert abs(loss - ref_loss) <= 1e-3 * ref_loss
    rel = np.linalg.norm(g - ref_g) / np.linalg.norm(ref_g)
    assert rel < 1e-2, rel
    assert losses[0] == loss
    # Adam's first step is lr g / (|g| + 1e-8) up to FP32 rounding of p
    step = p0 - p1
    want = 1e-3 * g / (np.abs(g) + 1e-8)
    assert np.abs(step - want).max() <= 1e-6 + 2 ** -23 * np.abs(p0).max()


def test_rows_do_not_depend_on_the_batch():
    """Every row's output is the same bits whichever rows come with it (4, 8
    or 16 rows per workgroup, full and ragged)."""
    widths = [5, 256, 130, 512]
    rng = np.random.default_rng(2)
    x = rng.uniform(-1, 1, size=(2100, 5)).astype(np.float32)
    with MLP(widths, max_batch=2100, seed=4) as net:
        whole = net.forward(x)
        for n in (1, 6, 1000, 1030, 2049):
            assert np.array_equal(net.forward(x[:n]), whole[:n]), n
        assert np.array_equal(net.forward(x[1000:1007]), whole[1000:1007])


def test_forward_without_copies():
    """Batches that go over pinned memory (to 4 MB) and beyond: a row's output
    does not depend on its batch, bit for bit."""
    rng = np.random.default_rng(8)
    x = rng.normal(size=(2100, 5))
    edge = (4 << 20) // (4 * (5 + 512))
    with MLP([5, 256, 256, 256, 256, 512], max_batch=2100) as m:
        want = m.forward(x)
        for batch in (1, 3, 128, edge, edge + 1):
            assert np.array_equal(m.forward(x[:batch]), want[:batch]), batch
        assert np.array_equal(m.forward(x[::-1][:77]), want[::-1][:77])  # a new batch in the same memory
