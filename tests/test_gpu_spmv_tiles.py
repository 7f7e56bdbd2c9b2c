"""The row tiles of 64, 128 and 512 rows at row counts around the choice
between them and with ragged last tiles, in the halo and the gather form,
with a long row and with contacts across tiles, against scipy in FP64: FP64
values 1e-13, FP32 values with FP32 tile copies 1e-6 (a few hundred 2^-24
roundings of mixed sign) relative."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def matrix(n, rng, long_row):
    """Upper BCOO of a band matrix (neighbours at 1, 2, 7) with far blocks; one row of n / 3 blocks when long_row."""
    i = np.concatenate([np.arange(n - k) for k in (0, 1, 2, 7) if k < n])
    j = np.concatenate([np.arange(k, n) for k in (0, 1, 2, 7) if k < n])
    a, b = rng.integers(0, n, (2, max(n // 10, 1)))
    if long_row:
        b = np.concatenate([b, rng.choice(n, n // 3, replace=False)])
        a = np.concatenate([a, np.full(n // 3, n // 2)])
    i, j = np.concatenate([i, np.minimum(a, b)]), np.concatenate([j, np.maximum(a, b)])
    key = np.unique(i.astype(np.int64) * n + j)
    r, c = (key // n).astype(np.int32), (key % n).astype(np.int32)
    v = rng.standard_normal((key.size, 3, 3))
    v[r == c] += v[r == c].transpose(0, 2, 1)
    k = np.arange(3)
    R, Cc = 3 * r[:, None, None] + k[None, :, None], 3 * c[:, None, None] + k[None, None, :]
    U = sp.coo_matrix((v.reshape(-1), (np.broadcast_to(R, v.shape).reshape(-1), np.broadcast_to(Cc, v.shape).reshape(-1))),
                      shape=(3 * n, 3 * n)).tocsr()
    d = r == c
    D = sp.coo_matrix((v[d].reshape(-1), (np.broadcast_to(R[d], v[d].shape).reshape(-1),
                                          np.broadcast_to(Cc[d], v[d].shape).reshape(-1))), shape=(3 * n, 3 * n)).tocsr()
    return np.ascontiguousarray(v.transpose(0, 2, 1)).reshape(-1, 9), r, c, (U + U.T - D)


@pytest.mark.parametrize("form", ["halo", "gather"])
@pytest.mark.parametrize("n,long_row", [(1, False), (65, False), (512, False), (513, False), (1000, True), (27999, False),
                                        (28000, True), (28127, False), (65535, False), (65537, True), (79999, False), (80000, False), (80513, True)])
def test_products(pkg, gpu_ctx, monkeypatch, form, n, long_row):
    monkeypatch.setenv("SGIPC_SPMV_GATHER", "1" if form == "gather" else "0")
    rng = np.random.default_rng(n)
    v, r, c, A = matrix(n, rng, long_row)
    ctx = gpu_ctx
    M = pkg.SpMat(ctx, ctx.to_device(v), ctx.to_device(r, np.int32), ctx.to_device(c, np.int32), r.size, n, want_f32=True)
    x, y0 = rng.standard_normal(3 * n), rng.standard_normal(3 * n)
    want = 0.7 * (A @ x) - 0.3 * y0
    for apply, tol in ((M.apply, 1e-13), (M.apply_f32_values, 1e-6)):
        y = ctx.to_device(y0)
        apply(0.7, ctx.to_device(x), -0.3, y)
        assert np.linalg.norm(y.download() - want) <= tol * np.linalg.norm(want)
    y = ctx.to_device(y0.astype(np.float32))
    M.apply(0.7, ctx.to_device(x.astype(np.float32)), -0.3, y)
    assert np.linalg.norm(y.download() - want) <= 1e-6 * np.linalg.norm(want)
    assert M.layout()[0] == (1 if form == "halo" else 0)
    assert M.long_rows() == (1 if long_row and n // 3 > 128 else 0)
    M.close()


@pytest.mark.parametrize("form", ["halo", "gather"])
@pytest.mark.parametrize("n,long_row", [(513, False), (1000, True), (27999, False), (28127, False), (60001, True)])
def test_small_tiles_sum_in_fp64(pkg, gpu_ctx, monkeypatch, form, n, long_row):
    """FP32 values against an FP64 vector, both exact in FP32: with the 64- and 128-row tiles' FP64 partial sums no
    rounding to FP32 is left, only a few hundred of 2^-53 of each row's absolute sum."""
    monkeypatch.setenv("SGIPC_SPMV_GATHER", "1" if form == "gather" else "0")
    rng = np.random.default_rng(n)
    v, r, c, _ = matrix(n, rng, long_row)
    f = v.astype(np.float32).astype(np.float64)
    x = rng.standard_normal(3 * n).astype(np.float32).astype(np.float64)
    H, d = f.reshape(-1, 3, 3).transpose(0, 2, 1), r == c
    k = np.arange(3)
    i, j = (np.broadcast_to(a, H.shape).reshape(-1) for a in (3 * r[:, None, None] + k[None, :, None],
                                                              3 * c[:, None, None] + k[None, None, :]))
    off = np.repeat(~d, 9)
    A = sp.coo_matrix((np.concatenate([H.reshape(-1), H.reshape(-1)[off]]),
                       (np.concatenate([i, j[off]]), np.concatenate([j, i[off]]))), shape=(3 * n, 3 * n)).tocsr()
    ctx = gpu_ctx
    M = pkg.SpMat(ctx, ctx.to_device(f), ctx.to_device(r, np.int32), ctx.to_device(c, np.int32), r.size, n, want_f32=True)
    y = ctx.to_device(np.zeros(3 * n))
    M.apply_f32_values(1.0, ctx.to_device(x), 0.0, y)
    M.close()
    err = (np.abs(y.download() - A @ x) / (abs(A) @ abs(x))).max()
    print(f"{form} {n} rows: {err:.1e} of the absolute sums")
    assert err <= 500 * 2.0 ** -53


@pytest.mark.parametrize("precision", ["fp64", "fp32_mas", "fp32_ir"])
@pytest.mark.parametrize("N,graph", [(9, True), (31, False)])
def test_default_iteration_folds_the_p_update(pkg, N, precision, graph):
    """On 64- and 128-row tiles the default iteration forms p inside the SpMV: the arithmetic of the separate update
    except for the grouping of two sums, so the iterates after 25 steps differ by amplified rounding only (the bound
    of the fused iteration's own test; 1e-6 where the tiles hold FP32 copies of p)."""
    ls = pkg.LinearSystem(pkg.scenes.tet_grid_scene("fold", N, n_pairs=8), bank_size=16)
    try:
        kw = dict(precision=precision, graph=graph, ir_replace_every=0)
        a = ls.solve(tol=1e-30, max_iter=26, fuse=1, **kw)
        b = ls.solve(tol=1e-30, max_iter=26, fuse=0, **kw)
        assert a.iterations == b.iterations
        assert np.linalg.norm(a.x - b.x) <= (1e-13 if precision != "fp32_ir" else 1e-6) * np.linalg.norm(b.x)
        a, b = (ls.solve(tol=1e-6, precision=precision, graph=graph, fuse=f) for f in (1, 0))
        assert abs(a.iterations - b.iterations) <= 1
        assert a.true_rel_residual <= 1e-6 and b.true_rel_residual <= 1e-6
    finally:
        ls.close()
