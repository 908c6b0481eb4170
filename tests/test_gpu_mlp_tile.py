"""Gradients of the training kernel at the edges of its tiles (32 records) and of its grid (512
workgroups, past which a workgroup takes several tiles), and the Adam steps built on them."""
import numpy as np
import pytest

from hcgpu import learned
from oracle import mlp_ref

pytestmark = pytest.mark.gpu


def _records(n, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((n, 8)).astype(np.float32)
    Y = np.stack([rng.standard_normal(n), (rng.random(n) < 0.4)], axis=1).astype(np.float32)
    W = np.stack([rng.random(n) < 0.8, np.ones(n)], axis=1).astype(np.float32)
    p = learned.init_params(seed) + 0.05 * rng.standard_normal(learned.NPARAMS).astype(np.float32)
    return p.astype(np.float32), X, Y, W


@pytest.mark.parametrize("n", [1, 15, 16, 31, 32, 33, 4096, 512 * 32, 512 * 32 + 1, 40001])
def test_gradient_matches_float64(gpu_ctx, n):
    p, X, Y, W = _records(n, n)
    pred, loss, grad = learned.forward_backward(gpu_ctx, p, X, Y, W)
    rl, rg, ro = mlp_ref.loss_and_grad(p, X.astype(np.float64), Y.astype(np.float64), W.astype(np.float64))
    # FP32 sums against FP64 sums of the same products: chains of at most 64 + 32 * tiles / 512 terms in
    # each accumulator, unit roundoff 6e-8, and GELU's few ulps; 1e-5 is about twenty times that
    np.testing.assert_allclose(pred, ro, rtol=1e-5, atol=1e-5)
    assert loss == pytest.approx(rl, rel=1e-5)
    assert np.linalg.norm(grad - rg) <= 1e-5 * np.linalg.norm(rg)


@pytest.mark.parametrize("n,batch", [(1, 1), (33, 32), (100, 4096)])
def test_one_epoch_of_adam(gpu_ctx, n, batch):
    """Every record once; the order of the records within an epoch is the library's, so batches of
    more than one step are compared through their loss."""
    p, X, Y, W = _records(n, 7 + n)
    q, _ = learned.train(gpu_ctx, p, X, Y, W, epochs=1, batch=batch, lr=1e-3, seed=3)
    if n <= batch:
        _, g, _ = mlp_ref.loss_and_grad(p, X.astype(np.float64), Y.astype(np.float64), W.astype(np.float64))
        step = 1e-3 * g / (np.abs(g) + 1e-8)  # Adam's first step
        big = np.abs(g) > 1e-5  # below, eps and FP32 rounding of the sum decide the step
        assert np.abs((p - q) - step)[big].max() <= 1e-5
    l0, l1 = (learned.forward_backward(gpu_ctx, v, X, Y, W)[1] for v in (p, q))
    assert l1 < l0
    again, _ = learned.train(gpu_ctx, p, X, Y, W, epochs=1, batch=batch, lr=1e-3, seed=3)
    np.testing.assert_array_equal(q, again)  # partial gradients are added in a fixed order
