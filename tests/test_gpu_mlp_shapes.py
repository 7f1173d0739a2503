"""The training kernels at the edges of their work split: batches around 64
rows (one workgroup's) and around the counts where the weight gradients are
dealt to 16, 8, 4, 2 or 1 workgroups, against the CPU restatement of the
network.  Tolerances as in test_gpu_mlp.py."""
import numpy as np
import pytest

from peridem_amd import capi
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 64, 65, 512, 1000, 1088, 4097, 8257])
def test_gradient_rows(rows):
    rng = np.random.default_rng(rows)
    net = capi.Mlp(seed=2)
    mean = rng.normal(size=16).astype(np.float32) * 0.1
    scale = rng.uniform(0.5, 2.0, size=16).astype(np.float32)
    osc, ow = np.array([1.0, 2.0, 0.5, 4.0], np.float32), np.array([1.0, 0.5, 2.0, 1.0], np.float32)
    net.set_normalization(mean, scale, osc, ow)
    x = rng.normal(size=(rows, 16)).astype(np.float32)
    t = rng.normal(size=(rows, 4)).astype(np.float32)
    loss, g = net.gradient(x, t)
    p = net.params().astype(np.float64)
    lr, gr = M.loss_and_grad(p, x, t, mean, scale, osc, ow)
    assert abs(loss - lr) <= 2e-3 * lr
    assert np.linalg.norm(g - gr) < 2e-2 * np.linalg.norm(gr)
    o = 0
    for s in M.SHAPES:
        k = int(np.prod(s))
        assert np.linalg.norm(g[o:o + k] - gr[o:o + k]) < 5e-2 * np.linalg.norm(gr[o:o + k]), s
        o += k
    y, yr = net.forward(x), M.predict(p, x, mean, scale, osc)
    assert np.abs(y - yr).max() < 1e-2 * np.abs(yr).max()
    # one training step moves every weight block the same way from the same draw
    a, b = capi.Mlp(seed=2), capi.Mlp(seed=2)
    for n in (a, b):
        n.train(x, t, iters=2, batch=rows, lr=1e-3, seed=3)
    np.testing.assert_array_equal(a.params(), b.params())
