"""Value sets that take turns on one grid: the path is captured once per
workspace and reads each run's values through a device pointer, and the
workspace keeps the largest capacities it has needed.  Every run must match
the oracle on its own values, whichever set ran before it and while another
result is alive."""
import numpy as np
import pytest

import support as S
import workloads as W
from test_gpu_pipeline_parity import _compare

pytestmark = pytest.mark.gpu


def _sets():
    rng = np.random.default_rng(77)
    many_small = W.mixed(rng, 0, 6, 0, 0)
    planes = W.mixed(rng, 6, 0, 0, 0)
    bundle = W.FuncSet()  # six planes through one point: tets with 5 and 6 functions, few with one
    for _ in range(6):
        bundle.plane([0.03, 0.02, -0.01], rng.standard_normal(3))
    return [many_small, planes, bundle]


@pytest.mark.parametrize("regular", [True, False])
def test_alternating_value_sets(ctx, regular):
    import rin

    res = 11
    pts, tets = S.grid(res)
    g = ctx.grid_regular(res) if regular else ctx.grid_explicit(pts, tets)
    sets = _sets()
    vals = [g.eval(*fs.arrays()) for fs in sets]
    refs = [S.OracleRun(0, pts, tets, S.evaluate(*fs.arrays(), pts)) for fs in sets]
    for i in (0, 1, 2, 0, 2, 1, 0, 1, 2):
        dev = vals[i].run(rin.FLAG_BATCHED)
        _compare(dev, refs[i])
        dev.release()
    # two results alive: the second run takes a workspace of its own
    a, b = vals[0].run(rin.FLAG_BATCHED), vals[1].run(rin.FLAG_BATCHED)
    _compare(a, refs[0])
    _compare(b, refs[1])
    # the values of a released set may come back at the same address with other contents
    a.release()
    vals[0].release()
    v = g.eval(*sets[2].arrays())
    c = v.run(rin.FLAG_BATCHED)
    _compare(c, refs[2])
    _compare(b, refs[1])
    for x in (c, b, v, vals[1], vals[2], g):
        x.release()
