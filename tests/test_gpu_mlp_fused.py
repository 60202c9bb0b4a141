"""The fused network kernels (256 hidden units) at the edges of their row tiles
(16, 32, 64, 128 rows), of the 32-row steps and splits of the weight gradients and of
their widths, against the CPU oracle. Tolerances as in test_gpu_mlp.py: a different
FP32 summation order moves values across a BF16 rounding boundary at a rate of about
1e-4, so outputs and gradients are compared in relative norm, 5e-3."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30)


def case(rows, n_in, n_out, seed=5):
    rng = np.random.default_rng(seed + rows)
    p = mo.init_params(n_in, 256, n_out, seed)
    p = (p + 0.02 * rng.normal(size=p.size)).astype(np.float32)
    return p, rng.normal(size=(rows, n_in)).astype(np.float32), rng.normal(size=(rows, n_out)).astype(np.float32)


def handle(n_in, n_out, max_batch, p):
    from cmf.surrogate import MLP
    g = MLP(max_batch=max_batch, n_in=n_in, n_out=n_out)
    g.set_params(p)
    return g


@pytest.mark.parametrize("rows, n_in, n_out", [(1, 24, 2), (15, 24, 2), (33, 32, 16), (130, 7, 1), (4096, 24, 2),
                                               (4097, 24, 2), (8193, 30, 3), (32769, 24, 2)])
def test_forward_and_gradient(rows, n_in, n_out):
    p, x, t = case(rows, n_in, n_out)
    g = handle(n_in, n_out, 40000, p)
    want_y = mo.forward(p, x, n_in, 256, n_out)[0]
    assert rel(g.forward(x), want_y) < 5e-3
    loss, grad = mo.loss_grad(p, x, t, n_in, 256, n_out)
    assert abs(g.grad(x, t) - loss) <= 5e-3 * loss
    assert rel(g.grads(), grad) < 5e-3
    # a smaller batch after a larger one sees none of its rows
    if rows > 100:
        loss, grad = mo.loss_grad(p, x[:19], t[:19], n_in, 256, n_out)
        assert abs(g.grad(x[:19], t[:19]) - loss) <= 5e-3 * loss
        assert rel(g.grads(), grad) < 5e-3
    g.close()


@pytest.mark.parametrize("batch", [16, 100, 1024])
def test_training_steps(batch):
    """Adam over gathered batches equals gradient calls on the same rows followed by
    the same update on the host, in relative norm of the parameter change."""
    p, x, t = case(3 * batch + 5, 24, 2, seed=9)
    g = handle(24, 2, 1024, p)
    hist = g.fit(x, t, 1, batch=batch, seed=4)
    got = g.params()
    order = np.random.default_rng(4).permutation(len(x))
    q, m1, m2, losses = p.astype(np.float64), 0.0, 0.0, []
    for k in range(3):
        i = order[k * batch:(k + 1) * batch]
        g.set_params(q.astype(np.float32))
        losses.append(g.grad(x[i], t[i]))
        d = g.grads().astype(np.float64)
        m1, m2 = 0.9 * m1 + 0.1 * d, 0.999 * m2 + 0.001 * d * d
        q = q - 1e-3 * (m1 / (1 - 0.9 ** (k + 1))) / (np.sqrt(m2 / (1 - 0.999 ** (k + 1))) + 1e-8)
    assert abs(hist[0] - np.mean(losses)) <= 1e-3 * np.mean(losses)
    # a gradient of a few ulps decides the sign of its Adam step: 2% in norm
    assert rel(got - p, (q - p)) < 0.02
    g.close()
