"""The patch search and the chain walk at their edges: a frontier wider than
the workgroup that walks a patch, faces of more corners than a neighbour row
holds, and chains that are cycles; against the reference's loops over the
device's faces."""
import math

import numpy as np
import pytest

import workloads as W
from test_gpu_edges import _chains_of, _patches_of

pytestmark = pytest.mark.gpu


def _functions(which):
    fs = W.FuncSet()
    if which == "wide":  # one plane: levels of more than 512 faces
        fs.plane([0.0, 0.0, 0.013], [0.11, 0.07, 1.0])
        return 160, fs
    if which == "corners":  # a polygon of nine sides or more inside the one cube's middle tet
        fs.plane([0.0, 0.0, 0.05], [0.0, 0.0, 1.0])
        for q in range(11):
            a = 0.1 + 2 * math.pi * q / 11
            n = [math.cos(a), math.sin(a), 0.02 * (q % 3)]
            fs.plane([0.12 * n[0], 0.12 * n[1], 0.05], n)
        return 1, fs
    # spheres that cross: cycles of non-manifold edges, short ones on the coarse grid
    for k in range(4):
        fs.sphere([0.3 * math.cos(k), 0.3 * math.sin(k), 0.1 * k], 0.45)
    return {"cycles": 24, "short": 4}[which], fs


@pytest.mark.parametrize("which", ["wide", "corners", "cycles", "short"])
def test_patches_and_chains(ctx, which):
    import rin

    res, fs = _functions(which)
    g = ctx.grid_regular(res)
    v = g.eval(*fs.arrays())
    dev = v.run(rin.FLAG_BATCHED)
    vs, fv, _, _, _ = dev.faces()
    corners = np.diff(vs.astype(np.int64))
    if which == "corners":
        assert corners.max() > 8
    start, faces = dev.patches()
    want = _patches_of(vs, fv)
    np.testing.assert_array_equal(np.diff(start.astype(np.int64)), [len(p) for p in want])
    np.testing.assert_array_equal(faces, np.concatenate(want))
    v12, es, occ, eof = dev.edges()
    cstart, cedges = dev.chains()
    chains = _chains_of(v12, np.diff(es.astype(np.int64)))
    np.testing.assert_array_equal(np.diff(cstart.astype(np.int64)), [len(c) for c in chains])
    np.testing.assert_array_equal(cedges, np.concatenate(chains) if chains else [])
    dev.release()
    v.release()
    g.release()
