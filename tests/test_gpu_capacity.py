"""Runs at the limits of the batched forms' workspaces.  RIN_RECORD_WORDS lowers
the record words that a run may take, so that small inputs reach the limit."""
import numpy as np
import pytest

import support as S
import workloads as W
from test_gpu_pipeline_parity import _compare

pytestmark = pytest.mark.gpu


def _values(mi, F, n, pts):
    """n of F planes through the box or near-equal materials; the others reach no tet."""
    rng = np.random.default_rng(90 + 10 * F + mi)
    fs = W.FuncSet()
    for _ in range(F):
        if mi:
            fs.sphere(rng.uniform(-0.1, 0.1, 3), rng.uniform(0.0, 0.02))
        else:
            fs.plane(rng.uniform(-0.5, 0.5, 3), rng.standard_normal(3))
    vals = S.evaluate(*fs.arrays(), pts)
    vals[:, n:] = -9.0 if mi else 1.0
    return vals


@pytest.mark.parametrize("mi,F", [(0, 8), (1, 20)])
@pytest.mark.parametrize("regular", [True, False])
def test_runs_after_a_growth_that_failed(ctx, monkeypatch, mi, F, regular):
    """A workspace that could not grow is not used as if it had."""
    import rin

    pts, tets = S.grid(3)
    g = ctx.grid_regular(3) if regular else ctx.grid_explicit(pts, tets)
    flags = rin.FLAG_BATCHED | (rin.FLAG_MI if mi else 0)
    sets = [_values(mi, F, n, pts) for n in (2, F)]
    refs = [S.OracleRun(mi, pts, tets, v) for v in sets]
    few, many = [g.upload(v) for v in sets]

    def check(v, ref):
        dev = v.run(flags)
        _compare(dev, ref)
        assert dev.stage_times()[0][0] == "batched path (one graph)"
        dev.release()

    check(few, refs[0])
    monkeypatch.setenv("RIN_RECORD_WORDS", "1000")
    with pytest.raises(rin.RinError):
        many.run(flags)
    check(few, refs[0])
    monkeypatch.delenv("RIN_RECORD_WORDS")
    check(many, refs[1])
    check(few, refs[0])
    for x in (few, many, g):
        x.release()
