"""Functions that vanish on vertices, edges and faces of a regular grid: the
lowest tets of a simplex's star need not hold its iso-vertex, so the vertex
dedup walks the star's later tets.  Small integer values make that the usual
case; the batched form must number every vertex as the oracle does."""
import numpy as np
import pytest

import support as S
from test_gpu_pipeline_parity import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,F,zeros", [(1, 1, 0.5), (1, 4, 0.7), (2, 3, 0.8), (3, 2, 0.3), (5, 3, 0.9), (8, 4, 0.6),
                                         (13, 2, 0.97)])
def test_zero_values_batched(ctx, res, F, zeros):
    import rin

    rng = np.random.default_rng(1000 * res + F)
    pts, tets = S.grid(res)
    vals = rng.integers(1, 4, (len(pts), F)) * rng.choice([-1.0, 1.0], (len(pts), F))
    vals[rng.random(vals.shape) < zeros] = 0.0
    ref = S.OracleRun(0, pts, tets, vals)
    g = ctx.grid_regular(res)
    v = g.upload(vals)
    dev = v.run(rin.FLAG_BATCHED)
    _compare(dev, ref)
    assert dev.stage_times()[0][0] == "batched path (one graph)"
    dev.release()
    v.release()
    g.release()


# One of these inputs differs from the oracle by one boundary face (276 for
# 275), in the plain and the batched form, and did so with every face compared
# by its vertex keys as well; why is not established.
KNOWN = pytest.mark.xfail(reason="one boundary face more than the oracle", strict=True)


@pytest.mark.parametrize("res,F,levels", [(1, 2, 2), (1, 5, 3), (2, 3, 2), pytest.param(3, 4, 4, marks=KNOWN), (5, 6, 5),
                                          (8, 3, 3), (6, 12, 40)])
@pytest.mark.parametrize("regular", [True, False])
def test_tied_materials(ctx, res, F, levels, regular):
    """Few distinct values: materials tie at vertices, along edges, on whole
    tet faces and tets, so boundary faces pair with other materials, corners
    are created lazily and more than once in a tet, and keys miss the star's
    lowest tets."""
    import rin

    rng = np.random.default_rng(7000 + 100 * res + F)
    pts, tets = S.grid(res)
    vals = rng.integers(0, levels, (len(pts), F)).astype(np.float64)
    ref = S.OracleRun(1, pts, tets, vals)
    g = ctx.grid_regular(res) if regular else ctx.grid_explicit(pts, tets)
    v = g.upload(vals)
    for flags in (rin.FLAG_BATCHED, rin.FLAG_BATCHED, 0):
        dev = v.run(rin.FLAG_MI | flags)
        _compare(dev, ref)
        dev.release()
    v.release()
    g.release()
