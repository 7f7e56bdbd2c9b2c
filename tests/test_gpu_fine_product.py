"""The fine product of the FP32 two-grid cycle: its FP32 row sums are amplified
at soft vertices next to stiff contacts, so they keep one order and one cut for
every matrix size.  A body's rows (whole 512-row tiles, whole domains of every
level, an exact coarse solve) beside other bodies that share no block with it
meet the same operations as alone -- what the others add are zeros -- so the
apply gives them the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def upper_rows(n, rng):
    """Neighbour CSR and upper BCOO of a chain of n vertices with links at 1 and 3."""
    i = np.concatenate([np.arange(n), np.arange(n - 1), np.arange(n - 3)])
    j = np.concatenate([np.arange(n), np.arange(1, n), np.arange(3, n)])
    o = np.lexsort((j, i))
    i, j = i[o], j[o]
    v = 0.2 * rng.uniform(-1.0, 1.0, (i.size, 3, 3))
    d = i == j
    v[d] = np.eye(3) * 10.0 ** rng.uniform(0.0, 2.0, (n, 1, 1)) * 2.0
    return v.transpose(0, 2, 1).reshape(-1, 9), i.astype(np.int32), j.astype(np.int32)


def neighbours(n, r, c):
    e = r != c
    a, b = np.concatenate([r[e], c[e]]), np.concatenate([c[e], r[e]])
    num = np.bincount(a, minlength=n)
    return (np.cumsum(num) - num).astype(np.uint32), num.astype(np.uint32), b[np.lexsort((b, a))].astype(np.uint32)


def apply(pkg, ctx, B, v, r, c, pairs, x, precision, solve=False):
    n = x.size // 3
    start, num, lst = neighbours(n, r, c)
    dev = [ctx.to_device(a, np.uint32) for a in (start, num, lst)]
    dv, dr, dc = ctx.to_device(v), ctx.to_device(r, np.int32), ctx.to_device(c, np.int32)
    mas = pkg.MASPreconditioner(ctx, B)
    try:
        mas.set_coarse_mode(2)
        mas.initPreconditioner_Neighbor(n, 0, lst.size, *dev)
        mas.initPreconditioner_Matrix()
        dp = ctx.to_device(pairs.reshape(-1), np.int32) if len(pairs) else None
        mas.setPreconditioner_bcoo(dv, dr, dc, r.size, 0, dp, len(pairs), precision)
        assert mas.level2_inverse() is not None
        z = ctx.empty(3 * n, np.float64)
        mas.preconditioning(ctx.to_device(x), z)
        z = z.download()
        if solve:
            # one iteration from zero: the iterate is alpha z
            y = ctx.empty(3 * n, np.float64)
            st = pkg.PCGSolver(ctx, tol=1e3, stop_mode=pkg.STOP_TRUE_RESIDUAL).solve(dv, dr, dc, r.size, n, mas,
                                                                                    ctx.to_device(x), y)
            return z, y.download(), st
        return z
    finally:
        mas.close()


def body(pkg, orc, N, pairs):
    s = pkg.scenes.tet_grid_scene(f"body{N}", N, E_loguniform=(1e4, 1e9), n_pairs=pairs)
    v, r, c = orc.assemble(s)
    return s, np.asarray(v).reshape(-1, 9), np.asarray(r), np.asarray(c)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("B", [16, 32])
@pytest.mark.parametrize("N,pairs", [(16, 0), (16, 800), (24, 1500), (32, 3000)])
def test_apply_of_a_body_beside_others(pkg, orc, gpu_ctx, B, N, pairs, precision):
    s, v, r, c = body(pkg, orc, N, pairs)
    rng = np.random.default_rng(N + B)
    m = 512 * 160                        # the other bodies' rows, past the last choice of a tile size
    w, p, q = upper_rows(m, rng)
    x, y = rng.standard_normal(3 * s.n), rng.standard_normal(3 * m)
    prec = pkg.FP64 if precision == "fp64" else pkg.FP32_MAS
    alone = apply(pkg, gpu_ctx, B, v, r, c, s.pairs, x, prec)
    beside = apply(pkg, gpu_ctx, B, np.concatenate([v, w]), np.concatenate([r, p + s.n]).astype(np.int32),
                   np.concatenate([c, q + s.n]).astype(np.int32), s.pairs, np.concatenate([x, y]), prec)[:3 * s.n]
    d = np.abs(alone - beside)
    print(f"{N}^3 B {B} {precision}: {np.linalg.norm(d) / np.linalg.norm(alone):.2e} in norm, "
          f"{d.max() / np.sqrt(np.mean(alone ** 2)):.2e} of the RMS")
    if precision == "fp32":
        np.testing.assert_array_equal(alone, beside)
    else:                                # FP64 row sums may be cut by the matrix size
        assert np.linalg.norm(d) <= 1e-9 * np.linalg.norm(alone)


@pytest.mark.parametrize("N,pairs", [(16, 800), (32, 3000)])
def test_solve_runs_the_same_cycle(pkg, orc, gpu_ctx, N, pairs):
    """Inside a PCG the cycle runs on the solver's matrix instead of the preconditioner's own: its first iterate is a
    multiple of the same z (to FP64 rounding of the sums that give the factor; an FP32 cycle of another cut is 1e-7 off)."""
    s, v, r, c = body(pkg, orc, N, pairs)
    x = np.random.default_rng(3).standard_normal(3 * s.n)
    z, y, st = apply(pkg, gpu_ctx, 32, v, r, c, s.pairs, x, pkg.FP32_MAS, solve=True)
    assert st.iterations == 1
    alpha = (y @ z) / (z @ z)
    assert np.max(np.abs(y - alpha * z)) <= 1e-13 * np.max(np.abs(y))
