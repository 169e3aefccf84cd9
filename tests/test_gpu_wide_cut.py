"""Tets with more than 8 active functions (or materials): the wavefront-a-tet
cut with the complex in LDS, the lane-a-tet cut behind it for complexes beyond
its capacities, and the -R check's counts in both insertion orders, against
the oracle."""
import numpy as np
import pytest

import support as S
import workloads as W
from test_gpu_pipeline_parity import _compare

pytestmark = pytest.mark.gpu


def _set(mi, F, spread, seed=0):
    rng = np.random.default_rng(100 * F + mi + seed)
    fs = W.FuncSet()
    for _ in range(F):
        if mi:  # near-equal materials: many compete in one tet
            fs.sphere(rng.uniform(-spread, spread, 3), rng.uniform(0.0, 0.02))
        else:
            fs.plane(rng.uniform(-spread, spread, 3), rng.standard_normal(3))
    return fs


# 24 planes: some tets outgrow the LDS complex (277 vertices)
CASES = [(0, 9, 0.8), (0, 12, 0.8), (0, 16, 0.9), (0, 24, 0.9), (1, 9, 0.1), (1, 20, 0.3), (1, 28, 0.1)]


@pytest.mark.parametrize("mi,F,spread", CASES)
@pytest.mark.parametrize("regular", [True, False])
def test_more_than_eight(ctx, mi, F, spread, regular):
    import rin

    res = 2
    pts, tets = S.grid(res)
    g = ctx.grid_regular(res) if regular else ctx.grid_explicit(pts, tets)
    fs = _set(mi, F, spread)
    vals = g.eval(*fs.arrays())
    ref = S.OracleRun(mi, pts, tets, S.evaluate(*fs.arrays(), pts))
    assert np.diff(ref.start_index.astype(np.int64)).max() > 8
    base = rin.FLAG_MI if mi else 0
    for flags in (0, rin.FLAG_NO_LOOKUP, rin.FLAG_BATCHED, rin.FLAG_BATCHED):
        dev = vals.run(base | flags)
        _compare(dev, ref)
        if flags == rin.FLAG_BATCHED and not mi:  # the batched form hands over what outgrows the LDS complex only
            assert (dev.stage_times()[0][0] == "batched path (one graph)") == (F < 24)
        dev.release()
    # another value set of the same plan, all of its tets with 8 functions or fewer
    few = S.evaluate(*fs.arrays(), pts)
    few[:, 8:] = -9.0 if mi else 1.0
    v2 = g.upload(few)
    dev = v2.run(base | rin.FLAG_BATCHED)
    _compare(dev, S.OracleRun(mi, pts, tets, few))
    dev.release()
    v2.release()
    vals.release()
    g.release()


@pytest.mark.parametrize("mi,F,spread", CASES)
@pytest.mark.parametrize("reverse", [False, True])
def test_counts_of_more_than_eight(ctx, mi, F, spread, reverse):
    import rin

    res = 2
    g = ctx.grid_regular(res)
    fs = _set(mi, F, spread)
    vals = g.eval(*fs.arrays())
    pts, tets = S.grid(res)
    hv = S.evaluate(*fs.arrays(), pts)
    ref = S.OracleRun(mi, pts, tets, hv)
    dev = vals.run((rin.FLAG_MI if mi else 0) | rin.FLAG_CUT_ONLY | (rin.FLAG_REVERSE if reverse else 0))
    got = dev.cut_counts()
    st = ref.start_index.astype(np.int64)
    for i, t in enumerate(ref.active.astype(np.int64)):
        rows = hv[tets[t].astype(np.int64)][:, ref.func_in_tet[st[t]:st[t + 1]].astype(np.int64)].T
        w = S.oracle_cut(mi, rows[::-1] if reverse else rows)
        assert tuple(got[i]) == (w[2], w[3], w[4])
    dev.release()
    vals.release()
    g.release()
