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


# edge and face counts around 16, 64 and 4096 (2, 5, 26), many more pairs than
# the first pair buffer and a workgroup's LDS hold (12 and 20 at a wide dhat),
# one flat axis, long thin sheets
CASES = {
    "tiny": dict(N=2), "small": dict(N=5), "tops": dict(N=26), "dense": dict(N=12, dhat=3e-3),
    "denser": dict(N=20, dhat=2.5e-3), "bodies": dict(N=9, body_ids=True),
}


def geometry(pkg, name):
    geo = pkg.scenes.contact_sheets(**CASES[name])
    if name == "tops":
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


@pytest.mark.parametrize("name", ["tiny", "small", "bodies", "dense"])
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
