"""The start network's training kernels at the edges of their tiling: one to four
input column tiles, one to twelve output column tiles, batches of one row tile, of a
whole fragment pass (32 row tiles) and beyond it.  Loss, gradient and forward
pass against the FP64 restatement with the same BF16 operand rounding (norm-wise
2e-3, the bar of FP32 against FP64 accumulation), and one Adam step against the
gradient it is made from.
"""
import numpy as np
import pytest

import accelerint_amd as acc
import mlp_ref

pytestmark = pytest.mark.gpu

SHAPES = [(1, 16), (5, 48), (14, 512), (15, 528), (46, 32), (54, 496), (62, 1040)]


def setup(n, B):
    rng = np.random.default_rng(31 * n + B)
    net = mlp_ref.Net(n)
    acc.mlp_init(n, 3)
    p = acc.mlp_params()
    x = rng.standard_normal((B, n + 2)).astype(np.float32)
    t = rng.standard_normal((B, 3 * n)).astype(np.float32)
    return net, p, x, t


@pytest.fixture
def session():
    acc.lib()
    yield acc
    acc.mlp_release()


@pytest.mark.parametrize("n,B", SHAPES)
def test_loss_gradient_and_forward(session, n, B):
    net, p, x, t = setup(n, B)
    loss, g = acc.mlp_loss_grad(x, t)
    L, G = net.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), bf=True)
    assert abs(loss - L) <= 2e-3 * L
    assert np.linalg.norm(g - G) <= 2e-3 * np.linalg.norm(G)
    y = acc.mlp_predict(x, 3 * n)
    # the loss of the forward pass's own outputs
    assert abs(((y.astype(np.float64) - t) ** 2).mean() - loss) <= 1e-5 * loss


@pytest.mark.parametrize("n,B", SHAPES)
def test_one_adam_step(session, n, B):
    net, p, x, t = setup(n, B)
    _, g = acc.mlp_loss_grad(x, t)
    lr = 1e-2
    hist = acc.mlp_train_host(x, t, 1, B, lr, seed=2)  # one batch: the samples in another order
    assert np.isfinite(hist).all()
    p1 = acc.mlp_params()
    # first step: lr g / (|g| + eps); gradients well above the summation order's rounding
    big = np.abs(g) > 1e-2 * np.abs(g).max()
    want = p - lr * g / (np.abs(g) + 1e-8)
    assert big.sum() > 20
    assert np.abs(p1 - want)[big].max() <= 1e-4 * lr + 4 * np.finfo(np.float32).eps * np.abs(p).max()
    # the operand tiles the step left behind are those of the new parameters
    y = acc.mlp_predict(x, 3 * n)
    acc.mlp_set_params(p1)
    assert np.array_equal(y, acc.mlp_predict(x, 3 * n))
