"""The tet kernel on both sides of the count from which it passes its blocks
through LDS wave by wave (20,000), at counts around a wave (64) and a workgroup
(128), with vertex ids in any order (blocks stored transposed) and gradients
whose vertices collide in the workgroup's table: against the oracle within 1e-10 of each element's largest
entry (the element arithmetic's rounding), the gradient within 1e-12
relative, with indices exact."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 63, 64, 65, 127, 128, 129, 300, 19999, 20000, 20031, 20032, 20033, 20096, 20097])
@pytest.mark.parametrize("spread", [False, True])
def test_tets(pkg, orc, gpu_ctx, m, spread):
    base = pkg.scenes.tet_grid_scene("waves", 6, E_loguniform=(1e4, 1e9))
    rng = np.random.default_rng(m)
    new = rng.permutation(base.n)
    # spread: the tets' vertices lie far apart in a larger vertex array
    ids = np.sort(rng.choice(100_000, base.n, replace=False)) if spread else np.arange(base.n)
    n = 100_000 if spread else base.n
    x = np.zeros((n, 3))
    x[ids[new]] = base.x
    pick = rng.choice(base.n_tets, m, replace=m > base.n_tets)
    tets = ids[new][base.tets[pick]].astype(np.int32)
    part = [np.ascontiguousarray(a[pick]) for a in (base.dm_inv, base.vol, base.mu, base.lam)]
    scene = dataclasses.replace(base, x=x, tets=tets, **dict(zip(("dm_inv", "vol", "mu", "lam"), part)))
    ov, orr, oc, og = orc.tet_snh(scene, hess_offset=5)
    c, L = gpu_ctx, pkg._lib.lib()
    dx, dt = c.to_device(x.reshape(-1)), c.to_device(tets.reshape(-1), np.uint32)
    dp = [c.to_device(a.reshape(-1)) for a in part]
    grad = c.to_device(np.zeros(3 * n))
    tv, tr, tc = c.empty((10 * m, 9), np.float64), c.empty(10 * m, np.int32), c.empty(10 * m, np.int32)
    pkg._lib.check(L.sgipc_fem_tet_gradient_hessian(c.h, dx.vp, dt.vp, *[d.vp for d in dp], m, base.dt, 5, grad.vp,
                                                    tv.vp, tr.vp, tc.vp), c.h)
    np.testing.assert_array_equal(tr.download(), orr)
    np.testing.assert_array_equal(tc.download(), oc)
    gv = tv.download().reshape(m, 90)
    ref = np.asarray(ov).reshape(m, 90)
    assert float((np.abs(gv - ref).max(1) / np.abs(ref).max(1)).max()) <= 1e-10
    g = grad.download()
    assert np.linalg.norm(g - np.asarray(og).reshape(-1)) <= 1e-12 * np.linalg.norm(og)
