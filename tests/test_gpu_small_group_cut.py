"""Tets of one and two functions without the lookup tables: groups of 8 lanes,
and the extraction's reads of four record words, against the oracle."""
import numpy as np
import pytest

import support as S
from test_gpu_pipeline_parity import _compare

pytestmark = pytest.mark.gpu


# tet counts below, at and past the 8 groups of a wavefront; ties (values of
# few levels, zeros among them) put corners, edges and faces on the planes
@pytest.mark.parametrize("res,F", [(2, 1), (2, 2), (3, 2), (7, 3), (9, 1)])
@pytest.mark.parametrize("levels", [0, 2])
@pytest.mark.parametrize("regular", [True, False])
def test_small_groups(ctx, res, F, levels, regular):
    import rin

    pts, tets = S.grid(res)
    rng = np.random.default_rng(10 * res + F)
    v = rng.uniform(-1, 1, (len(pts), F))
    if levels:
        v = np.round(v * levels) / levels
    g = ctx.grid_regular(res) if regular else ctx.grid_explicit(pts, tets)
    vals = g.upload(v)
    ref = S.OracleRun(0, pts, tets, v)
    for flags in (rin.FLAG_NO_LOOKUP, 0):
        dev = vals.run(flags)
        _compare(dev, ref)
        dev.release()
    for reverse in (False, True):
        dev = vals.run(rin.FLAG_CUT_ONLY | (rin.FLAG_REVERSE if reverse else 0))
        got = dev.cut_counts()
        st = ref.start_index.astype(np.int64)
        for i in range(0, len(ref.active), 1 + len(ref.active) // 64):
            t = int(ref.active[i])
            rows = v[tets[t].astype(np.int64)][:, ref.func_in_tet[st[t]:st[t + 1]].astype(np.int64)].T
            w = S.oracle_cut(0, rows[::-1] if reverse else rows)
            assert tuple(got[i]) == (w[2], w[3], w[4])
        dev.release()
    vals.release()
    g.release()
