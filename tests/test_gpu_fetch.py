"""Results to host memory in packed chunks: streams of exactly one chunk, one
word more, chunks shared by several arrays, and long ones that several host
threads copy.  Uploaded values come back bit for bit, and the arrays of a mesh
that spans many chunks agree with each other."""
import numpy as np
import pytest

import workloads as W

pytestmark = pytest.mark.gpu


# one chunk is 262144 words: 64^3 vertices of one function
@pytest.mark.parametrize("res,F", [(1, 1), (63, 1), (64, 1), (63, 2), (64, 3), (63, 8), (64, 9)])
def test_values_round_trip(ctx, res, F):
    g = ctx.grid_regular(res)
    rng = np.random.default_rng(res * 100 + F)
    a = rng.standard_normal(((res + 1) ** 3, F))
    a[0, 0] = np.nan
    a[-1, -1] = -0.0
    v = g.upload(a)
    np.testing.assert_array_equal(v.download().view(np.uint64), a.view(np.uint64))
    v.release()
    g.release()


def test_many_chunks_agree(ctx):
    """At 97^3 vertices the CSR is 17 chunks, the vertices and faces about ten."""
    import rin

    res = 96
    g = ctx.grid_regular(res)
    fs = W.mixed(np.random.default_rng(5), 3, 3, 1, 1)
    v = g.eval(*fs.arrays())
    hv = v.download()
    dev = v.run(rin.FLAG_BATCHED)
    s = dev.sizes
    fit, start = dev.csr()
    assert start[0] == 0 and start[-1] == s.n_func_in_tet == len(fit)
    k = np.diff(start.astype(np.int64))
    assert np.count_nonzero(k) == s.num_intersecting and fit.max() < len(fs)
    # the active functions of a sample of tets, by their corner values
    import support as S

    _, tets = S.grid(res)
    for t in np.random.default_rng(6).integers(0, len(tets), 4000):
        c = hv[tets[t].astype(np.int64)]
        want = [f for f in range(len(fs)) if not ((c[:, f] > 0).all() or (c[:, f] < 0).all())]
        assert list(fit[start[t]:start[t + 1]]) == want
    rec, xyz = dev.verts()
    none = np.uint64(2 ** 64 - 1)
    size = rec[:, 2].astype(np.int64)
    assert size.min() >= 1 and size.max() <= 4 and np.abs(xyz).max() <= 1.0
    np.testing.assert_array_equal((rec[:, 3:7] != none).sum(axis=1), size)
    np.testing.assert_array_equal((rec[:, 7:11] != none).sum(axis=1), size - 1)
    vs, fv, ts, tf, fn = dev.faces()
    assert vs[-1] == len(fv) and ts[-1] == len(tf) and fv.max() == len(rec) - 1
    assert (k[tf[:, 0].astype(np.int64)] > 0).all() and (fn[:, 0] < len(fs)).all() and (fn[:, 1] == none).all()
    # every vertex of a face carries the face's function
    f0 = np.repeat(fn[:, 0], np.diff(vs.astype(np.int64)))
    assert (rec[fv.astype(np.int64), 7:11] == f0[:, None]).any(axis=1).mean() > 0.999
    dev.release()
    v.release()
    g.release()
