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


@pytest.mark.parametrize("res,F,levels", [(1, 2, 2), (1, 5, 3), (2, 3, 2), (3, 4, 4), (5, 6, 5), (8, 3, 3),
                                          (6, 12, 40)])
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


def _six_tets(res):
    """res^3 cubes of six tets around the main diagonal."""
    n = res + 1
    i, j, k = np.meshgrid(*[np.arange(res)] * 3, indexing="ij")
    base = ((i * n + j) * n + k).reshape(-1)
    step = [n * n, n, 1]
    tets = []
    for p, even in (((0, 1, 2), 1), ((1, 2, 0), 1), ((2, 0, 1), 1), ((0, 2, 1), 0), ((2, 1, 0), 0), ((1, 0, 2), 0)):
        a = base + step[p[0]]
        b = a + step[p[1]]
        c = b + step[p[2]]
        tets.append(np.stack([base, a, b, c] if even else [base, b, a, c], -1))
    ax = np.linspace(-1.0, 1.0, n)
    return np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3), np.stack(tets, 1).reshape(-1, 4)


@pytest.mark.parametrize("mesh", ["regular", "six tets", "tets permuted", "vertices permuted"])
def test_materials_tied_across_a_face(ctx, mesh):
    """Materials that tie on a whole tet face name its vertices differently from
    its two sides; the reference then tells the two copies of a boundary face
    apart by their least, second and greatest vertex ids, which on an edge go
    by the first of the tets around it.  Small meshes of few values, until
    the case has come up many times."""
    import rin

    rng = np.random.default_rng(["regular", "six tets", "tets permuted", "vertices permuted"].index(mesh))
    for _ in range(25):
        res, F, levels = int(rng.integers(2, 6)), int(rng.integers(3, 8)), int(rng.integers(3, 5))
        pts, tets = _six_tets(res) if mesh == "six tets" else S.grid(res)
        if mesh == "tets permuted":
            tets = tets[rng.permutation(len(tets))]
        if mesh == "vertices permuted":
            p = rng.permutation(len(pts))
            pts, tets = pts[np.argsort(p)], p[tets.astype(np.int64)]
        tets = np.ascontiguousarray(tets.astype(np.uint64))
        pts = np.ascontiguousarray(pts)
        vals = rng.integers(0, levels, (len(pts), F)).astype(np.float64)
        ref = S.OracleRun(1, pts, tets, vals)
        g = ctx.grid_regular(res) if mesh == "regular" else ctx.grid_explicit(pts, tets)
        v = g.upload(vals)
        for flags in (rin.FLAG_BATCHED, 0):
            dev = v.run(rin.FLAG_MI | flags)
            _compare(dev, ref)
            dev.release()
        v.release()
        g.release()
