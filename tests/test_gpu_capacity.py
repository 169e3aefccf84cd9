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
    """A run past the limit takes the plain form, and a workspace that could not
    grow is not used as if it had."""
    import rin

    pts, tets = S.grid(3)
    g = ctx.grid_regular(3) if regular else ctx.grid_explicit(pts, tets)
    flags = rin.FLAG_BATCHED | (rin.FLAG_MI if mi else 0)
    sets = [_values(mi, F, n, pts) for n in (2, F)]
    refs = [S.OracleRun(mi, pts, tets, v) for v in sets]
    few, many = [g.upload(v) for v in sets]

    def check(v, ref, path="batched path (one graph)"):
        dev = v.run(flags)
        _compare(dev, ref)
        assert dev.stage_times()[0][0].startswith(path)
        dev.release()

    check(few, refs[0])
    monkeypatch.setenv("RIN_RECORD_WORDS", "1000")
    check(many, refs[1], "batched form fell back")
    check(few, refs[0])
    monkeypatch.delenv("RIN_RECORD_WORDS")
    check(many, refs[1])
    check(few, refs[0])
    for x in (few, many, g):
        x.release()


# record words of a slot by the tet's functions: 2, 3..4, 5..8, 9..28
SLOTS = ((2, 2, 324), (3, 4, 952), (5, 8, 4536), (9, 28, 13248))


@pytest.mark.parametrize("regular", [True, False])
def test_wide_tets_leave_the_other_slots_alone(ctx, monkeypatch, regular):
    """A value set with tets of nine functions, then one of five to eight in most
    tets, under a limit that both fit when only the former have large slots."""
    import rin

    pts, tets = S.grid(5)
    g = ctx.grid_regular(5) if regular else ctx.grid_explicit(pts, tets)
    rng = np.random.default_rng(3)
    fs = W.FuncSet()
    for _ in range(9):
        fs.plane(rng.uniform(-0.02, 0.02, 3) + [0.1, 0.05, 0.0], rng.standard_normal(3))
    wide = S.evaluate(*fs.arrays(), pts)
    many = rng.integers(1, 4, (len(pts), 9)) * rng.choice([-1.0, 1.0], (len(pts), 9))
    many[:, 8] = 1.0
    refs = [S.OracleRun(0, pts, tets, v) for v in (wide, many)]
    k = [np.diff(r.start_index.astype(np.int64)) for r in refs]
    assert k[0].max() == 9 and k[1].max() == 8
    n = [max(int(((x >= lo) & (x <= hi)).sum()) for x in k) for lo, hi, _ in SLOTS]
    assert n[3] < 20 and n[2] > 400
    need = sum((x + 64) * 9 // 8 * w for x, (_, _, w) in zip(n, SLOTS))
    assert (n[2] + 64) * 9 // 8 * SLOTS[3][2] > 1.5 * need  # as one list with the larger slots
    monkeypatch.setenv("RIN_RECORD_WORDS", str(int(1.1 * need)))
    values = [g.upload(v) for v in (wide, many)]
    for i in (0, 1, 0, 1):
        dev = values[i].run(rin.FLAG_BATCHED)
        _compare(dev, refs[i])
        assert dev.stage_times()[0][0] == "batched path (one graph)"
        dev.release()
        dev = values[i].run(rin.FLAG_BATCHED | rin.FLAG_STAGE_TIMES)  # the same launches, a graph a stage
        _compare(dev, refs[i])
        assert "cut k=9.. (wave per tet)" in [n for n, _ in dev.stage_times()]
        dev.release()
    for v in values:
        v.release()
    g.release()


@pytest.mark.parametrize("regular", [True, False])
def test_more_functions_than_the_cut_takes(ctx, regular):
    """Value sets of one plan in turn: tets of 9..28 functions, of at most 8, and
    of more than 28; the last give the plain form's error each time."""
    import rin

    pts, tets = S.grid(4)
    g = ctx.grid_regular(4) if regular else ctx.grid_explicit(pts, tets)
    rng = np.random.default_rng(5)
    fs = W.FuncSet()
    for _ in range(32):
        fs.plane([0.1, 0.05, 0.0], rng.standard_normal(3))
    too_many = S.evaluate(*fs.arrays(), pts)
    wide, few = too_many.copy(), too_many.copy()
    wide[:, 9:] = 1.0
    few[:, 7:] = 1.0
    active = [(~((v[tets.astype(int)] > 0).all(1) | (v[tets.astype(int)] < 0).all(1))).sum(1).max()
              for v in (too_many, wide, few)]
    assert active[0] > 28 and 8 < active[1] <= 28 and 4 < active[2] <= 8
    values = {n: g.upload(v) for n, v in (("wide", wide), ("few", few), ("too many", too_many))}
    refs = {"wide": S.OracleRun(0, pts, tets, wide), "few": S.OracleRun(0, pts, tets, few)}
    with pytest.raises(rin.RinError) as plain:
        values["too many"].run(0)
    for n in ("too many", "few", "too many", "wide", "too many", "few", "wide"):
        if n == "too many":
            with pytest.raises(rin.RinError) as e:
                values[n].run(rin.FLAG_BATCHED)
            assert str(e.value) == str(plain.value)
            continue
        dev = values[n].run(rin.FLAG_BATCHED)
        _compare(dev, refs[n])
        assert dev.stage_times()[0][0] == "batched path (one graph)"
        dev.release()
    for v in values.values():
        v.release()
    g.release()


@pytest.mark.parametrize("mi,F,res", [(0, 12, 50), (1, 12, 62)])
def test_record_words_past_32_bits(ctx, mi, F, res):
    """Most tets with more than 8 functions: their record slots' words pass 2^32,
    and the run is refused before anything of their size is allocated."""
    import rin

    pts, tets = S.grid(res)
    rng = np.random.default_rng(6)
    vals = rng.uniform(-1.0, 1.0, (len(pts), F))
    if mi:
        vals[:, :] = rng.permuted(np.tile(np.arange(F, dtype=np.float64), (len(pts), 1)), axis=1)
        c = vals[tets.astype(int)]  # a lower bound of a tet's materials: each corner's highest, and the rule's
        top = c.argmax(2)
        low = np.stack([np.take_along_axis(c[:, q], top, 1).min(1) for q in range(4)], 1)
        active = ((c > low[:, :, None]).sum(1) > 1)
        np.put_along_axis(active, top, True, 1)
        k, words = active.sum(1), 7928
    else:
        c = vals[tets.astype(int)]
        k, words = (~((c > 0).all(1) | (c < 0).all(1))).sum(1), 13248
    assert k.max() <= 28 and int((k > 8).sum()) * words > 1 << 32
    g = ctx.grid_regular(res)
    v = g.upload(vals)
    for flags in (rin.FLAG_BATCHED, 0, rin.FLAG_NO_LOOKUP):
        with pytest.raises(rin.RinError, match="record slots exceed"):
            v.run(flags | (rin.FLAG_MI if mi else 0))
    v.release()
    g.release()
