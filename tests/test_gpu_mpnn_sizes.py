"""Training kernels of the learned level at node and row counts around their
tiles (4 nodes per gather workgroup, 32 per layer tile, 256-row and 384-row
chunks, 8 XCD runs), against the numpy oracle with the same bf16 operands.
With the identity activation no term switches, so what is left is the order of
FP32 sums and the few operands it moves across a bf16 rounding boundary (one
part in 256 of single operands, averaged over a row's 128): 5e-3 of each
parameter block, 1e-3 of the loss."""
import numpy as np
import pytest

from oracle import mpnn

pytestmark = pytest.mark.gpu


def chain_operator(n, rng):
    """A symmetric positive definite block operator: neighbours at 1, 2 and n // 2, so rows differ in length."""
    import scipy.sparse as sp
    i = np.arange(n)
    e = np.unique(np.sort(np.concatenate([np.stack([i[:-k], i[k:]], 1) for k in {1, 2, max(n // 2, 1)} if k < n]
                                         or [np.zeros((0, 2), int)]), axis=1), axis=0)
    A = sp.lil_matrix((3 * n, 3 * n))
    for a, b in e:
        d = rng.standard_normal(3)
        K = np.outer(d, d) + 0.1 * np.eye(3)
        for p, q, s in ((a, a, 1), (b, b, 1), (a, b, -1), (b, a, -1)):
            A[3 * p:3 * p + 3, 3 * q:3 * q + 3] += s * K
    return (A + 0.5 * sp.eye(3 * n)).tocsr()


@pytest.mark.parametrize("n,samples", [(1, 1), (3, 2), (32, 1), (33, 3), (85, 1), (86, 5), (130, 9)])
def test_loss_and_gradient(pkg, gpu_ctx, n, samples):
    rng = np.random.default_rng(n + samples)
    A = chain_operator(n, rng)
    graph = mpnn.coarse_graph(A, np.arange(n), n)
    v, r, c = mpnn.coarse_upper_bcoo(graph.A1, n)
    data = pkg.learned.MpnnData.from_bcoo(gpu_ctx, n, v, r, c)
    X = rng.standard_normal((samples, 3 * n, 3)).astype(np.float32)
    q = np.ascontiguousarray(X[:, :, 2])
    data.add(X, q)
    net = pkg.learned.Mpnn(gpu_ctx, layers=2, linear=True)
    p = mpnn.init_params(64, 2, seed=3)
    net.set_params(p.flat())
    loss, g = net.loss_grad(data, 0, samples)
    want, pg = mpnn.loss_grad(mpnn.Params.from_flat(net.get_params(), 64, 2), graph.Ahat,
                              [(X[k].astype(np.float64), q[k].astype(np.float64)) for k in range(samples)],
                              bf16_ops=True, linear=True)
    got = mpnn.Params.from_flat(g, 64, 2)
    assert abs(loss - want) <= 1e-3 * abs(want)
    for a, b in ((got.W_in, pg.W_in), (got.W[0], pg.W[0]), (got.W[1], pg.W[1]), (got.w_out, pg.w_out)):
        assert np.linalg.norm(a - b) <= 5e-3 * np.linalg.norm(b)
    net.close()
    data.close()
