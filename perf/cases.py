"""The calls whose speed this repository measures: the per-tet arrangement and
interface path through its public entry points (rin.Context, grids, values,
runs and the result accessors), over the sizes, forms and options that its
configurations, its tests and its serving stream use.

listed() names the cases and draw() gives others of the same ranges;
prepare() makes what a program has before the call (a context and a grid that
it keeps, and function values or function descriptors from a seed), run() does
one pass, work() says what a pass cannot do without, tolerance() how far two
correct results may be apart."""
import ctypes
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "robust-implicit-surface-networks_amd"))
import rin  # noqa: E402
import workloads  # noqa: E402

# What a case's fields say:
#   mode       "ia" (implicit arrangement) or "mi" (material interface)
#   res        cubes a side; the regular grid has (res + 1)^3 vertices and 5 res^3 tets
#   mesh       "regular", or "explicit": a jittered mesh of 6 res^3 tets as a file would hold it
#   functions  how many functions (or materials)
#   kind       "mixed" (planes, spheres, cylinders and tori 6:6:4:4), "spheres", "dyadic" (planes on
#              grid coordinates and through grid vertices, two functions twice: exact zeros and ties
#              everywhere) or "materials" (-|x - p| + w)
#   form       "batched", "plain" (one launch a stage) or "general" (lookup tables off)
#   take       what the program does with the result:
#              "resident"  the mesh stays on the GPU, as in the benchmark's step
#              "host"      vertices and faces come to host memory
#              "dropin"    all that implicit_arrangement() takes: CSR, vertices, faces, iso-edges,
#                          patches and chains
#              "job"       a served request: functions evaluated on the grid, the run, the mesh to host
#              "robust"    the -R check: complex counts per tet, forward and reversed


def _case(name, mode, res, functions, kind, form="batched", take="resident", mesh="regular"):
    return {"name": name, "mode": mode, "res": res, "functions": functions, "kind": kind, "form": form, "take": take,
            "mesh": mesh}


def listed():
    return [
        # the smallest configuration (3 planes and 2 spheres' size of problem): launches and latency
        _case("ia_20_f5_host", "ia", 20, 5, "mixed", take="host"),
        # the benchmark's step: 101^3 vertices, 20 functions, mesh left on the GPU
        _case("ia_100_f20", "ia", 100, 20, "mixed"),
        # the same, taken to the host as a caller of the library does
        _case("ia_100_f20_host", "ia", 100, 20, "mixed", take="host"),
        # the finest grid: four times the tets of the paper's largest, fewer functions
        _case("ia_200_f8", "ia", 200, 8, "mixed"),
        # the drop-in's device calls at the paper's smallest grid, four spheres
        _case("ia_45_f4_dropin", "ia", 45, 4, "spheres", take="dropin"),
        # degenerate input: exact predicates and ties decide
        _case("ia_32_dyadic18", "ia", 32, 18, "dyadic"),
        # the lookup-table ablation: every tet through the general cut
        _case("ia_99_f18_general", "ia", 99, 18, "spheres", form="general"),
        # a mesh from a file: explicit tets, an odd size
        _case("ia_explicit_37_f6_host", "ia", 37, 6, "mixed", take="host", mesh="explicit"),
        # the robustness check's two cut passes
        _case("ia_49_f8_robust", "ia", 49, 8, "mixed", form="plain", take="robust"),
        # a served request with the most functions the stream has
        _case("job_32_f32", "ia", 32, 32, "mixed", take="job"),
        # the material-interface configuration, mesh left on the GPU
        _case("mi_64_m8", "mi", 64, 8, "materials"),
        # the paper's largest material-interface run, taken to the host
        _case("mi_99_m18_host", "mi", 99, 18, "materials", take="host"),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case: grid and function count spread over the range of its
    family, odd sizes among them."""
    f = rng.choice(["resident", "resident", "host", "dropin", "dyadic", "general", "explicit", "robust", "job", "mi",
                    "mi"])
    if f == "resident":
        res = _log(rng, 16, 200)
        most = max(1, min(32, int(20e6 / res ** 3)))
        return _draw("ia", res, _log(rng, 1, max(2, most)), rng.choice(["mixed", "spheres"]))
    if f == "host":
        res = _log(rng, 16, 100)
        return _draw("ia", res, rng.randint(1, 20), "mixed", take="host")
    if f == "dropin":
        return _draw("ia", _log(rng, 20, 64), rng.randint(2, 12), rng.choice(["mixed", "spheres"]), take="dropin")
    if f == "dyadic":
        return _draw(rng.choice(["ia", "mi"]), rng.choice([16, 32, 64]), rng.randint(6, 18), "dyadic",
                     take=rng.choice(["resident", "host"]))
    if f == "general":
        return _draw(rng.choice(["ia", "mi"]), _log(rng, 20, 99), rng.randint(2, 18), "spheres",
                     form=rng.choice(["plain", "general"]))
    if f == "explicit":
        return _draw(rng.choice(["ia", "mi"]), _log(rng, 8, 40), rng.randint(2, 12), "spheres",
                     take=rng.choice(["resident", "host"]), mesh="explicit")
    if f == "robust":
        return _draw(rng.choice(["ia", "mi"]), _log(rng, 12, 49), rng.randint(2, 8), "spheres", form="plain",
                     take="robust")
    if f == "job":
        mode = rng.choice(["ia", "ia", "mi"])
        return _draw(mode, rng.choice([16, 32, 64]), rng.randint(2, 32), "mixed" if mode == "ia" else "materials",
                     form="batched" if mode == "ia" else "plain", take="job")
    return _draw("mi", _log(rng, 16, 99), rng.randint(2, 18), "materials", take=rng.choice(["resident", "host"]))


def _draw(*a, **k):
    c = _case("", *a, **k)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs


def _functions(case, seed):
    """Function descriptors of a case, from the seed alone."""
    rng = np.random.default_rng(seed)
    n, kind = case["functions"], case["kind"]
    if kind == "mixed":
        part = [0.3, 0.3, 0.2, 0.2]
        c = [int(n * p) for p in part]
        for i in range(n - sum(c)):
            c[i % 4] += 1
        fs = workloads.mixed(rng, *c)
    elif kind == "spheres":
        fs = workloads.mixed(rng, 0, n, 0, 0)
    elif kind == "materials":
        fs = workloads.FuncSet()
        for _ in range(n):
            fs.sphere(rng.uniform(-0.8, 0.8, 3), rng.uniform(0.0, 0.2))
    else:
        # two thirds axis-aligned planes on grid coordinates, then planes
        # through three grid vertices with integer normals, then two repeats
        half = case["res"] // 2
        fs = workloads.FuncSet()
        axis_planes = max(1, 2 * n // 3)
        for j in range(axis_planes):
            pt, nrm = [0.0] * 3, [0.0] * 3
            pt[j % 3] = int(rng.integers(2 - half, half - 1)) / half
            nrm[j % 3] = 1.0
            fs.plane(pt, nrm)
        while len(fs) < n - 2:
            P = rng.integers(-half, half + 1, size=(3, 3)) / half
            nrm = np.cross(P[1] - P[0], P[2] - P[0]) * half * half
            if np.any(nrm):
                fs.plane(P[0], nrm)
        while len(fs) < n:
            fs.copy_of(int(rng.integers(0, len(fs))))
        fs = fs.permuted(rng.permutation(n))
    return fs.arrays()


def _jittered(res):
    """A tet mesh as a file would hold it: res^3 cubes of six tets around the
    main diagonal, inner vertices moved by up to a fifth of the spacing."""
    n = res + 1
    axis = np.linspace(-1.0, 1.0, n)
    pts = np.stack(np.meshgrid(axis, axis, axis, indexing="ij"), -1).reshape(-1, 3)
    inner = np.all(np.abs(pts) < 1.0 - 1e-9, axis=1)
    rng = np.random.default_rng(7)
    pts[inner] += rng.uniform(-0.2, 0.2, (int(inner.sum()), 3)) * (2.0 / res)
    i, j, k = np.meshgrid(*[np.arange(res)] * 3, indexing="ij")
    base = ((i * n + j) * n + k).reshape(-1)
    step = [n * n, n, 1]
    tets = []
    for p, even in (((0, 1, 2), 1), ((1, 2, 0), 1), ((2, 0, 1), 1), ((0, 2, 1), 0), ((2, 1, 0), 0), ((1, 0, 2), 0)):
        a = base + step[p[0]]
        b = a + step[p[1]]
        c = b + step[p[2]]
        tets.append(np.stack([base, a, b, c] if even else [base, b, a, c], -1))
    return pts, np.stack(tets, 1).reshape(-1, 4)


class _Program:
    """What a program keeps for one mesh: its context, the mesh on the GPU and
    the one result that it works with (the next run replaces it)."""

    def __init__(self, mesh, res):
        self.ctx = rin.Context(0)
        self.grid = self.ctx.grid_regular(res) if mesh == "regular" else self.ctx.grid_explicit(*_jittered(res))
        self.results = []

    def keep(self, *results):
        self.results = list(results)
        return results[0]

    def drop(self):
        for r in self.results:
            r.release()
        self.results = []

    def __del__(self):
        if getattr(self, "grid", None) is not None:
            self.drop()
            self.grid.release()
            self.ctx.close()


class _State:
    def __init__(self, program, case, types, params):
        self.program, self.case, self.types, self.params = program, case, types, params
        self.vals = None if case["take"] == "job" else program.grid.eval(types, params)
        # the caller's buffers, as the C ABI fills them
        self.buffers = {} if case["take"] == "resident" else {k: _buffers(case, k) for k in _TAKES[case["take"]]}

    def __del__(self):
        if getattr(self, "vals", None) is not None:
            self.vals.release()


# ------------------------------------------------------------------ the caller's buffers

_TAKES = {"resident": ["csr", "verts", "faces"], "host": ["verts", "faces"], "job": ["verts", "faces"],
          "dropin": ["csr", "verts", "faces", "edges", "patches", "chains"], "robust": ["forward", "reversed"]}


def _buffers(case, what):
    """Buffers for one accessor, large enough for any functions of the case
    (a mesh takes a fifth of them or more; what lies behind its end stays zero)."""
    F, sq = case["functions"], case["res"] ** 2
    nv = int(((6.0 * F if case["mode"] == "ia" else 10.0 * F ** 0.5) + 12.0) * sq) + 64 * case["res"]
    nt = (5 if case["mesh"] == "regular" else 6) * case["res"] ** 3
    nf, corners = 5 * nv // 2, 7 * nv
    sizes = {"csr": [3 * nv, nt + 1], "verts": [(nv, 11), (nv, 3)],
             "faces": [nf + 1, corners, nf + 1, (3 * nv, 2), (nf, 2)],
             "edges": [(4 * nv, 2), 4 * nv + 1, (corners, 2), corners], "patches": [nf + 1, nf],
             "chains": [nv + 1, 4 * nv], "forward": [(2 * nv, 3)], "reversed": [(2 * nv, 3)]}[what]
    got = [np.zeros(n, dtype=np.uint64) for n in sizes]
    if what == "verts":
        got[1] = got[1].view(np.float64)
    return got


def _p(a):
    return a.ctypes.data_as(rin._f64p if a.dtype == np.float64 else rin._u64p)


def _read(result, what, bufs):
    """One accessor's arrays into the caller's buffers; the numbers of their rows in use."""
    L, ctx, s = rin.lib(), result.ctx, result.sizes
    n = ctypes.c_uint64(0)
    if what == "csr":
        used, call = [s.n_func_in_tet, s.n_tets + 1], L.rin_result_csr
    elif what == "verts":
        used, call = [s.n_verts, s.n_verts], L.rin_result_verts
    elif what == "faces":
        used, call = [s.n_faces + 1, s.n_face_verts, s.n_faces + 1, s.n_tet_faces, s.n_faces], L.rin_result_faces
    elif what == "edges":
        ctx.check(L.rin_result_edge_count(ctx.h, result.h, ctypes.byref(n)))
        used, call = [n.value, n.value + 1, s.n_face_verts, s.n_face_verts], L.rin_result_edges
    elif what == "patches":
        ctx.check(L.rin_result_patch_count(ctx.h, result.h, ctypes.byref(n)))
        used, call = [n.value + 1, s.n_faces], L.rin_result_patches
    elif what == "chains":
        ctx.check(L.rin_result_edge_count(ctx.h, result.h, ctypes.byref(n)))
        edges = n.value
        ctx.check(L.rin_result_chain_count(ctx.h, result.h, ctypes.byref(n)))
        used, call = [n.value + 1, edges], L.rin_result_chains
    else:
        used, call = [s.num_intersecting], L.rin_result_cut_counts
    for u, b in zip(used, bufs):
        if u > len(b):
            raise RuntimeError("%s: %d rows and a buffer of %d" % (what, u, len(b)))
    ctx.check(call(ctx.h, result.h, *[_p(b) for b in bufs]))
    return used


_program = (None, None)  # the mesh in use now, and its program


def prepare(case, seed):
    global _program
    key = (case["mesh"], case["res"])
    if _program[0] != key:
        _program = (None, None)  # the last mesh goes before the next comes
        _program = (key, _Program(*key))
    return _State(_program[1], case, *_functions(case, seed))


# ------------------------------------------------------------------ a pass


class _OnGpu(dict):
    """A result's mesh where the run leaves it, on the GPU: its arrays come to
    the host when they are looked at, by the accessors that a program would call."""

    def __init__(self, case, result):
        super().__init__((k, None) for k in _TAKES["resident"])
        self.case, self.result = case, result

    def __getitem__(self, what):
        bufs = _buffers(self.case, what)
        return [_read(self.result, what, bufs), bufs]


_FORM = {"batched": rin.FLAG_BATCHED, "plain": 0, "general": rin.FLAG_NO_LOOKUP}


def run(state):
    c, p, B = state.case, state.program, state.buffers
    flags = _FORM[c["form"]] | (rin.FLAG_MI if c["mode"] == "mi" else 0)
    p.drop()
    if c["take"] == "resident":
        return _OnGpu(c, p.keep(state.vals.run(flags)))
    if c["take"] == "robust":
        flags |= rin.FLAG_CUT_ONLY
        a, b = state.vals.run(flags), state.vals.run(flags | rin.FLAG_REVERSE)
        p.keep(a, b)
        return [_read(a, "forward", B["forward"]), _read(b, "reversed", B["reversed"]), B]
    if c["take"] == "job":
        # as the server runs a request: evaluated values, the usual kernels without tuning
        vals = p.grid.eval(state.types, state.params)
        r = p.keep(vals.run(flags | (rin.FLAG_FIXED_FORMS if c["form"] == "batched" else 0)))
    else:
        vals = None
        r = p.keep(state.vals.run(flags | (rin.FLAG_KEEP_RECORDS if c["take"] == "dropin" else 0)))
    used = [_read(r, what, B[what]) for what in _TAKES[c["take"]]]
    if vals is not None:
        p.drop()
        vals.release()
    return [used, B]


# ------------------------------------------------------------------ what a pass needs


def work(case):
    """Values read once (a job writes them first) and outputs written once: the
    CSR's offsets, and the mesh at its usual size: 59 bytes a vertex, and on
    the host 112."""
    res, F = case["res"], case["functions"]
    V = (res + 1) ** 3
    T = (5 if case["mesh"] == "regular" else 6) * res ** 3
    # vertices per function and grid square, as counted over some seeds (materials: per root of their number)
    if case["mode"] == "ia":
        verts = {"mixed": 3.0, "spheres": 2.1, "dyadic": 1.5}.get(case["kind"], 3.0) * F * res * res
    else:
        verts = 4.5 * F ** 0.5 * res * res
    faces, corners, tets = 1.6 * verts, 5.3 * verts, 1.4 * verts
    b = 8.0 * F * V + (16.0 * T if case["mesh"] == "explicit" else 0.0)
    take = case["take"]
    if take == "job":
        b += 8.0 * F * V
    if take == "robust":
        return {"bytes": 2 * (b + 24.0 * tets), "flops": 0.0}
    device = verts * 59 + faces * 16 + corners * 4 + 4.0 * T + tets
    b += device
    if take in ("host", "dropin", "job"):
        b += verts * 112 + faces * 52 + corners * 8
    if take == "dropin":
        b += 8.0 * (T + tets) + corners * (8 * 3 + 12) + faces * 8
    return {"bytes": b, "flops": 0.0}


def tolerance(case):
    """Signs are exact and coordinates follow one stated order of operations
    without fused multiply-adds, so every result is the same to the bit."""
    return "exact"


def exact(case, seed):
    """No counterpart: the rows of a mesh are in the order in which this
    library's per-tet complexes list them, and the coordinates are the same to
    the bit."""
    return None
