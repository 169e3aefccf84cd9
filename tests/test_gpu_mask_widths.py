"""Function counts at the edges of the sign-mask widths (8, 16, 32 and 64
bits), grids whose last cube tile and rank block are partial, and the records
of single tets (found through the rank blocks), against the oracle."""
import numpy as np
import pytest

import support as S
import workloads as W
from test_gpu_pipeline_parity import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,F", [(1, 1), (2, 8), (7, 9), (5, 16), (9, 17), (6, 32), (8, 33), (4, 64)])
@pytest.mark.parametrize("regular", [True, False])
def test_mask_widths(ctx, res, F, regular):
    import rin

    rng = np.random.default_rng(10 * res + F)
    fs = W.mixed(rng, 0, F, 0, 0)
    pts, tets = S.grid(res)
    vals = S.evaluate(*fs.arrays(), pts)
    # few functions a tet: the rest of each set stays positive there
    vals += rng.uniform(0.0, 0.02, vals.shape)
    if F > 8:
        vals[:, rng.permutation(F)[6:]] = np.abs(vals[:, rng.permutation(F)[6:]]) + 0.5
        vals[:, F - 1] = pts[:, 0] - 0.013  # the highest bit of the masks is in use
    ref = S.OracleRun(0, pts, tets, vals)
    g = ctx.grid_regular(res) if regular else ctx.grid_explicit(pts, tets)
    v = g.upload(vals)
    dev = v.run(rin.FLAG_BATCHED | rin.FLAG_KEEP_RECORDS)
    _compare(dev, ref)
    pick = rng.integers(0, len(tets), 50).astype(np.uint64)
    st, w = dev.records(pick)
    row = {int(t): i for i, t in enumerate(ref.active)}
    for i, t in enumerate(pick):
        got = w[int(st[i]):int(st[i + 1])]
        if int(t) not in row:
            assert len(got) == 0
        else:
            a = row[int(t)]
            np.testing.assert_array_equal(got, ref.words[int(ref.rec_start[a]):int(ref.rec_start[a + 1])])
    dev.release()
    v.release()
    g.release()
