"""The restriction of a MAS apply (key sums within 16- and 32-lane groups, the
coarse levels in one workgroup from 1024 nodes down) against sums formed from
the apply's own tables and inverse blocks: interleaved chains give one, several
or a full domain of nodes per domain, and level-1 counts on both sides of the
1024 nodes.  The level sums, the solves (rows of at most 96 products) and the
sum over the levels are FP64 in another order: at most 96 + 64 + 8 roundings of
2^-53 on terms whose absolute sum is the bound below; 1e-5 for FP32, with
2^-24 in their place."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def chains(n, k, rng):
    """Neighbour CSR and diagonally dominant upper BCOO of k interleaved chains."""
    i = np.arange(n - k)
    nb = np.stack([np.arange(n) - k, np.arange(n) + k], 1)
    ok = (nb >= 0) & (nb < n)
    num = ok.sum(1).astype(np.uint32)
    start = (np.cumsum(num) - num).astype(np.uint32)
    r = np.concatenate([np.arange(n), i]).astype(np.int32)
    c = np.concatenate([np.arange(n), i + k]).astype(np.int32)
    v = rng.uniform(-1, 1, (r.size, 3, 3))
    v[:n] = v[:n] + v[:n].transpose(0, 2, 1) + 12 * np.eye(3)
    order = np.lexsort((c, r))
    nbr = nb[ok].astype(np.uint32)
    return (start, num, nbr if nbr.size else np.zeros(1, np.uint32)), v.transpose(0, 2, 1).reshape(-1, 9)[order], \
        r[order], c[order]


@pytest.mark.parametrize("precision", ["fp64", "fp32_mas"])
@pytest.mark.parametrize("B,n,k", [(16, 65, 1), (16, 257, 16), (16, 1024 * 16, 1), (16, 1024 * 16 + 1, 1),
                                   (16, 1023 * 8, 2), (32, 4099, 32), (32, 1024 * 32 + 7, 1), (32, 1025 * 4 - 3, 8)])
def test_apply_equals_its_levels(pkg, gpu_ctx, B, n, k, precision):
    ctx, rng = gpu_ctx, np.random.default_rng(n + k)
    (start, num, lst), v, r, c = chains(n, k, rng)
    dev = [ctx.to_device(a, np.uint32) for a in (start, num, lst)]
    mats = (ctx.to_device(v), ctx.to_device(r, np.int32), ctx.to_device(c, np.int32))
    mas = pkg.MASPreconditioner(ctx, B)
    try:
        mas.initPreconditioner_Neighbor(n, 0, int(num.sum()), *dev)
        mas.initPreconditioner_Matrix()
        mas.setPreconditioner_bcoo(*mats, r.size, 0, None, 0, pkg.FP64 if precision == "fp64" else pkg.FP32_MAS)
        x = rng.standard_normal((n, 3))
        dz = ctx.empty(3 * n, np.float64)
        mas.preconditioning(ctx.to_device(x.reshape(-1)), dz)
        z = dz.download().reshape(n, 3)
        L, off, cnt, total = mas.levels()
        ct, _ = mas.tables()
        inv = mas.inverse_blocks()
    finally:
        mas.close()
    iu, ju = np.triu_indices(B)
    dense = np.zeros((inv.shape[0], B, 3, B, 3))
    h = inv.reshape(inv.shape[0], iu.size, 3, 3)
    dense[:, iu, :, ju, :] = h.transpose(1, 0, 3, 2)
    dense[:, ju, :, iu, :] = h.transpose(1, 0, 2, 3)
    dense = dense.reshape(-1, 3 * B, 3 * B)
    want, size = np.zeros((n, 3)), np.zeros((n, 3))
    for l in range(L):
        slot = np.arange(n) if l == 0 else ct[:, l - 1]
        g, ga = np.zeros((total, 3)), np.zeros((total, 3))
        np.add.at(g, slot, x)
        np.add.at(ga, slot, np.abs(x))
        y = np.einsum("dij,dj->di", dense, g.reshape(-1, 3 * B)).reshape(-1, 3)
        ya = np.einsum("dij,dj->di", np.abs(dense), ga.reshape(-1, 3 * B)).reshape(-1, 3)
        want += y[slot]
        size += ya[slot]
    eps = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    assert np.all(np.abs(z - want) <= 170 * eps * size)
