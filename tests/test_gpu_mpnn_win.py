"""The gradient of the input weights over some 100k rows against a 64-bit sum.
With zero layer and input weights and the identity activation the output is
zero, so the gradient is sum over rows of X[row][g] * (-q[row] / rows) * w_out[c]
with one FP32 factor per row that holds no rounding but that of 1 / rows.  A
wave adds 24 rows in FP32 (multiply-adds), four waves' sums follow and FP64
from there: at most 24 + 4 + 1 roundings of 2^-24 of the absolute sum.  One
large term in 64 rows makes a longer chain lose the small ones behind it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,samples", [(1024, 32), (1021, 33)])
def test_input_weight_gradient(pkg, gpu_ctx, n, samples):
    C, L = pkg.learned.CHANNELS, 1
    rng = np.random.default_rng(n)
    i = np.arange(n - 1)
    r, c = np.concatenate([np.arange(n), i]), np.concatenate([np.arange(n), i + 1])
    o = np.lexsort((c, r))
    v = np.where((r == c)[:, None, None], 4.0, -1.0) * np.eye(3)
    data = pkg.learned.MpnnData.from_bcoo(gpu_ctx, n, v.reshape(-1, 9)[o], r[o].astype(np.int32), c[o].astype(np.int32))
    rows = 3 * n * samples
    X = np.ones((rows, 3), np.float32)
    X[np.arange(rows) % 256 < 4] = 2.0 ** 24
    X[:, 2] = rng.standard_normal(rows)
    q = -np.ones(rows, np.float32)
    data.add(X.reshape(samples, 3 * n, 3), q.reshape(samples, 3 * n))
    net = pkg.learned.Mpnn(gpu_ctx, layers=L, linear=True)
    w_out = 2.0 ** rng.integers(-3, 4, C)
    net.set_params(np.concatenate([np.zeros(3 * C + L * 2 * C * C), w_out]).astype(np.float32))
    _, g = net.loss_grad(data, 0, samples)
    net.close()
    data.close()
    x, scale = X.astype(np.float64), np.float64(np.float32(1.0) / np.float32(rows))
    err = np.abs(g[:3 * C].reshape(3, C) - scale * np.outer(x.sum(0), w_out)) / (scale * np.outer(np.abs(x).sum(0), w_out))
    print(f"{rows} rows: {err.max() * 2 ** 24:.1f} units of 2^-24")
    assert err.max() <= 29 * 2.0 ** -24
