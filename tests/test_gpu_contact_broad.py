"""The broad phase's clusters of 64 primitives, queries of 16 and tops of 4096
at the sizes and orders where they can go wrong, against the brute-force
oracle: pairs, MatIndex and counts bit-exact, the CCD step within 1e-9
(conservative advancement, its last step's rounding) with equal candidates."""
import ctypes
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def shuffled(geo, seed):
    """The same surface with vertices, faces, edges and surface slots in random order."""
    rng = np.random.default_rng(seed)
    new = rng.permutation(geo.n)          # old id -> new id
    inv = np.argsort(new)
    faces, edges = (new[a][rng.permutation(len(a))].astype(np.int32) for a in (geo.faces, geo.edges))
    return dataclasses.replace(geo, x=geo.x[inv], rest=geo.rest[inv], faces=faces, edges=edges,
                               surf=rng.permutation(geo.n).astype(np.int32),
                               body_id=None if geo.body_id is None else geo.body_id[inv])


# counts around 16 and 64 (2, 5), just past 4096 edges (27: 4160), faces (35:
# 4624) and points (46: 4232), so that a set spans several tops, many more pairs
# than the first pair buffer and a workgroup's LDS hold (12 and 20 at a wide
# dhat), one flat axis, long thin sheets
CASES = {
    "tiny": dict(N=2), "small": dict(N=5), "dense": dict(N=12, dhat=3e-3), "denser": dict(N=20, dhat=2.5e-3),
    "bodies": dict(N=9, body_ids=True), "edge_tops": dict(N=27), "face_tops": dict(N=35), "point_tops": dict(N=46),
}


def geometry(pkg, name):
    geo = pkg.scenes.contact_sheets(**CASES[name])
    if name.endswith("tops"):
        assert max(len(geo.edges), len(geo.faces), geo.n) > 4096
        x = geo.x.copy()
        x[:, 0] *= 30.0                   # long thin triangles
        geo = dataclasses.replace(geo, x=x)
    return shuffled(geo, 7)


@pytest.mark.parametrize("name", list(CASES))
def test_detection_of_shuffled_surfaces(pkg, orc, gpu_ctx, name):
    geo = geometry(pkg, name)
    want, wmi, wc = orc.contact_detect(geo.x, geo.rest, geo.faces, geo.edges, geo.surf, geo.dhat ** 2,
                                       body_id=geo.body_id)
    up = lambda a, t: gpu_ctx.to_device(np.ascontiguousarray(a).reshape(-1), t)
    body = up(geo.body_id, np.int32) if geo.body_id is not None else None
    det = pkg.ContactDetector(gpu_ctx)
    pairs, mi, counts = det.detect(up(geo.x, np.float64), up(geo.rest, np.float64), up(geo.faces, np.uint32),
                                   len(geo.faces), up(geo.edges, np.uint32), len(geo.edges), up(geo.surf, np.uint32),
                                   geo.surf.size, geo.n, geo.dhat ** 2, body_id=body)
    n = int(counts[0])
    print(f"{name}: {n} pairs of {geo.n} vertices")
    np.testing.assert_array_equal(counts, wc)
    np.testing.assert_array_equal(pairs.download()[:n], want)
    np.testing.assert_array_equal(mi.download()[:n], wmi)


@pytest.mark.parametrize("name", ["tiny", "small", "bodies", "dense", "edge_tops", "face_tops", "point_tops"])
def test_ccd_of_shuffled_surfaces(pkg, orc, gpu_ctx, name):
    geo = geometry(pkg, name)
    rng = np.random.default_rng(11)
    d = rng.uniform(-1e-4, 1e-4, geo.x.shape)
    d[geo.rest[:, 2] > 0, 2] += 6e-4
    want, nc = orc.ccd_self_step(geo.x, d, 1.0, geo.faces, geo.edges, geo.surf, geo.dhat ** 2, 0.8,
                                 body_id=geo.body_id)
    L, h = pkg._lib.lib(), gpu_ctx.h
    up = lambda a, t: gpu_ctx.to_device(np.ascontiguousarray(a).reshape(-1), t)
    body = up(geo.body_id, np.int32) if geo.body_id is not None else None
    x, dd, f, e, s = (up(geo.x, np.float64), up(d, np.float64), up(geo.faces, np.uint32), up(geo.edges, np.uint32),
                      up(geo.surf, np.uint32))
    step, cnt = ctypes.c_double(), ctypes.c_int()
    pkg._lib.check(L.sgipc_ccd_self_step(h, x.vp, dd.vp, 1.0, f.vp, len(geo.faces), e.vp, len(geo.edges), s.vp,
                                         geo.surf.size, body.vp if body else None, None, geo.dhat ** 2, 0.8,
                                         ctypes.byref(step), ctypes.byref(cnt)), h)
    assert cnt.value == nc
    assert step.value == pytest.approx(want, rel=1e-9)


def copies(geo, K):
    """K copies of the surface 2^-2 apart on a cubic grid.  Coordinates are multiples of 2^-40 below 16, so every
    difference of two is exact and each copy meets the arithmetic of the first."""
    grid = lambda a: np.round(a * 2.0 ** 40) / 2.0 ** 40
    x, rest = grid(geo.x), grid(geo.rest)
    side = int(np.ceil(K ** (1 / 3)))
    k = np.arange(K)
    at = 0.25 * np.stack([k % side, k // side % side, k // side ** 2], 1)
    all_of = lambda a: (a[None] + geo.n * k.reshape(-1, *([1] * a.ndim))).reshape(-1, *a.shape[1:]).astype(np.int32)
    return dataclasses.replace(geo, x=x, rest=rest), dataclasses.replace(
        geo, x=(x[None] + at[:, None]).reshape(-1, 3), rest=(rest[None] + at[:, None]).reshape(-1, 3),
        faces=all_of(geo.faces), edges=all_of(geo.edges), surf=all_of(geo.surf))


def test_more_than_64_tops(pkg, orc, gpu_ctx):
    """920 copies of a shuffled sheet pair far from one another: 65 tops of points, 109 of faces and 173 of edges.  Every pair
    is one of the oracle's pairs of a single copy, and the step is that of a single copy."""
    K = 920
    one, geo = copies(shuffled(pkg.scenes.contact_sheets(12), 5), K)
    assert min(geo.n, len(geo.faces), len(geo.edges)) > 64 * 4096
    det = lambda g, e: orc.contact_detect(g.x, g.rest, g.faces, e, g.surf, g.dhat ** 2)
    base = det(one, one.edges)[0]
    n_vf = len(det(one, one.edges[:0])[0])
    # ids moved by copy: entry 0 is -vertex - 1 (a vertex where two edges meet inside), entries 2 and 3 may be
    # absent (-1), entry 3 may be -edge - 2 (nearly parallel edges)
    copy = np.arange(K)[:, None]
    nv, ne = one.n * copy, len(one.edges) * copy
    move = lambda p: np.stack([np.where(p[:, 0] < 0, p[:, 0] - nv, p[:, 0] + nv), p[:, 1] + nv,
                               np.where(p[:, 2] < 0, -1, p[:, 2] + nv),
                               np.where(p[:, 3] < -1, p[:, 3] - ne, np.where(p[:, 3] < 0, -1, p[:, 3] + nv))], 2).reshape(-1, 4)
    want = np.concatenate([move(base[:n_vf]), move(base[n_vf:])])
    cls = np.where(want[:, 0] >= 0, 4, np.where(want[:, 2] < 0, 2, np.where(want[:, 3] < 0, 3, 4)))
    wmi = np.zeros(len(want), np.int64)
    for c in (2, 3, 4):
        wmi[cls == c] = np.arange((cls == c).sum())
    up = lambda a, t: gpu_ctx.to_device(np.ascontiguousarray(a).reshape(-1), t)
    x, f, e, s = up(geo.x, np.float64), up(geo.faces, np.uint32), up(geo.edges, np.uint32), up(geo.surf, np.uint32)
    pairs, mi, counts = pkg.ContactDetector(gpu_ctx).detect(x, up(geo.rest, np.float64), f, len(geo.faces), e,
                                                            len(geo.edges), s, geo.surf.size, geo.n, geo.dhat ** 2)
    n = int(counts[0])
    print(f"{K} copies: {n} pairs of {geo.n} vertices")
    assert list(counts) == [len(want), 0] + [int((cls == c).sum()) for c in (2, 3, 4)]
    np.testing.assert_array_equal(pairs.download()[:n], want)
    np.testing.assert_array_equal(mi.download()[:n], wmi)
    d = np.round(np.random.default_rng(11).uniform(-1e-4, 1e-4, one.x.shape) * 2.0 ** 40) / 2.0 ** 40
    d[one.rest[:, 2] > 0, 2] += 2.0 ** -11
    step, nc = orc.ccd_self_step(one.x, d, 1.0, one.faces, one.edges, one.surf, one.dhat ** 2, 0.8)
    got, cnt = ctypes.c_double(), ctypes.c_int()
    dd = up(np.tile(d, (K, 1)), np.float64)
    pkg._lib.check(pkg._lib.lib().sgipc_ccd_self_step(
        gpu_ctx.h, x.vp, dd.vp, 1.0, f.vp, len(geo.faces), e.vp, len(geo.edges), s.vp, geo.surf.size, None, None,
        geo.dhat ** 2, 0.8, ctypes.byref(got), ctypes.byref(cnt)), gpu_ctx.h)
    assert cnt.value == K * nc
    assert got.value == pytest.approx(step, rel=1e-9)
