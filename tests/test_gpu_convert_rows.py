"""The conversion by row counting at the row lengths where its paths change
(a wave's 64, 128 and 256 triplets, a workgroup's 2048, the common sort of the
longer rows, the general conversion when these hold more than half of the
triplets), with blocks of more and fewer than 64 triplets: values bit-exact
against the oracle (the order of the sums is part of the result), indices,
counts and status codes equal."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def convert(pkg, ctx, v, r, c, cap):
    L = pkg._lib.lib()
    dv, dr, dc = ctx.to_device(v), ctx.to_device(r, np.int32), ctx.to_device(c, np.int32)
    ov, orr, oc = (ctx.to_device(a) for a in (np.full((max(cap, 1), 9), 7.0), np.full(max(cap, 1), -7, np.int32),
                                              np.full(max(cap, 1), -7, np.int32)))
    nnz = ctypes.c_int()
    st = L.sgipc_convert_srbk(ctx.h, dv.vp, dr.vp, dc.vp, r.size, ov.vp, orr.vp, oc.vp, cap, ctypes.byref(nnz))
    return st, nnz.value, ov.download(), orr.download(), oc.download()


def triplets(lengths, width, rng):
    """Row i gets lengths[i] triplets over `width` columns at or past it, the rows' triplets mixed."""
    r = np.repeat(np.arange(len(lengths)), lengths).astype(np.int32)
    r = r[rng.permutation(r.size)]
    c = (r + rng.integers(0, width, r.size)).astype(np.int32)
    v = rng.standard_normal((r.size, 9)) * 10.0 ** rng.integers(-6, 7, (r.size, 1))
    return v, r, c


ROWS = {
    "waves": ([0, 1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 0, 500, 3], 40),
    "chunks": ([64, 65, 128, 129, 200, 256], 1),
    "long_blocks": ([300, 2000, 4000, 64], 2),
    "mid": ([2047, 2048, 2049, 700, 12], 600),
    "long": ([16383, 16384, 100], 5000),
    "too_long": ([16385, 30, 0, 9], 300),
    "few_rows": ([9000], 3),
    "some_long": ([2049, 30, 5000, 2048] + [40] * 2000 + [3000], 700),
    "long_one_block": ([9000] + [90] * 1000, 1),
    "long_last": ([20] * 3000 + [4097, 2500], 30000),
    "share_below": ([20000] + [25] * 800, 100),
    "share_above": ([20001] + [25] * 800, 100),
    "many_long": ([2100] * 40 + [64] * 12000, 3000),
    "long_wide_blocks": ([5000, 4100, 3] + [60] * 400 + [2600], 20),
    "many_short": (list(np.random.default_rng(1).integers(0, 90, 3000)), 12),
}


@pytest.mark.parametrize("name", list(ROWS))
def test_matches_oracle(pkg, orc, gpu_ctx, name):
    lengths, width = ROWS[name]
    v, r, c = triplets(lengths, width, np.random.default_rng(len(name)))
    want = orc.convert(v, r, c)
    n = want[1].size
    st, nnz, ov, orr, oc = convert(pkg, gpu_ctx, v, r, c, n + 3)
    assert (st, nnz) == (0, n)
    np.testing.assert_array_equal(orr[:n], want[1])
    np.testing.assert_array_equal(oc[:n], want[2])
    np.testing.assert_array_equal(ov[:n], np.asarray(want[0]).reshape(-1, 9))
    assert (ov[n:] == 7.0).all() and (orr[n:] == -7).all()
    # too small an output: the count needed, and nothing past the capacity
    st, nnz, ov, orr, oc = convert(pkg, gpu_ctx, v, r, c, n - 1)
    assert (st, nnz) == (pkg._lib.SGIPC_CAPACITY, n)
    np.testing.assert_array_equal(orr[:n - 1], want[1][:n - 1])


def test_bad_index(pkg, gpu_ctx):
    v, r, c = triplets([300] * 50, 9, np.random.default_rng(0))
    for k, (a, b) in enumerate([(-1, 3), (5, 4)]):
        rr, cc = r.copy(), c.copy()
        rr[77 + k], cc[77 + k] = a, b
        assert convert(pkg, gpu_ctx, v, rr, cc, r.size)[0] == pkg._lib.SGIPC_BAD_INDEX


def test_one_far_index(pkg, orc, gpu_ctx):
    """Few triplets and a large index: more rows than the row tables are worth."""
    v, r, c = triplets([5, 9, 2], 4, np.random.default_rng(3))
    c[4] = 5_000_000
    want = orc.convert(v, r, c)
    st, nnz, ov, orr, oc = convert(pkg, gpu_ctx, v, r, c, r.size)
    assert (st, nnz) == (0, want[1].size)
    np.testing.assert_array_equal(ov[:nnz], np.asarray(want[0]).reshape(-1, 9))
    np.testing.assert_array_equal(oc[:nnz], want[2])
