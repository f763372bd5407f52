"""The work that programs have this framework do, as cases that can be timed.

Most of it is adapt(): a box mesh and a target metric go in, the adapted mesh
comes out.  The listed cases take it from the smallest meshes, where launches
and waits count, to the 64^3 level-set box that bench.py times, with each kind
of metric (isotropic and anisotropic, 2D and 3D), growing and shrinking
meshes, tags carried along, the mixed-precision form and many small meshes at
once; the rest are the steps around it: building the box, preparing its
metric, and measuring lengths and qualities on device arrays.

Data that already lives on the GPU stays there: inputs and outputs of the
array entry points are torch tensors, handed over as device pointers.
"""
import ctypes
import math

import numpy as np
import torch

import omega_h_amd as A
from omega_h_amd import workloads as W

_ctx = None


def _context():
    """A program keeps one context for as long as it runs."""
    global _ctx
    if _ctx is None:
        _ctx = A.Context(0)
    return _ctx


def listed():
    return [
        # the shortest request of a server: a handful of tets, all latency
        {"name": "adapt3d_tiny", "kind": "adapt", "dim": 3, "n": 3, "metric": "constant",
         "elems": 300, "aspect": 1.5, "precision": 0},
        # the 2D workload of the benchmark: 2048 triangles, isotropic ring
        {"name": "adapt2d_ring", "kind": "adapt", "dim": 2, "n": 32, "metric": "ring",
         "elems": 0, "aspect": 1.0, "precision": 0},
        # a 2D request of a server: anisotropic constant metric, odd size
        {"name": "adapt2d_aniso", "kind": "adapt", "dim": 2, "n": 75, "metric": "constant",
         "elems": 40000, "aspect": 3.0, "precision": 0},
        # a 3D request that mostly refines: a coarse box grows tenfold
        {"name": "adapt3d_growth", "kind": "adapt", "dim": 3, "n": 9, "metric": "constant",
         "elems": 30000, "aspect": 2.0, "precision": 0},
        # an ordinary level-set adaptation, odd size
        {"name": "adapt3d_level_25", "kind": "adapt", "dim": 3, "n": 25, "metric": "levelset",
         "elems": 0, "aspect": 1.0, "precision": 0},
        # the benchmark's headline: 1,572,864 tets around a level set
        {"name": "adapt3d_level_64", "kind": "adapt", "dim": 3, "n": 64, "metric": "levelset",
         "elems": 0, "aspect": 1.0, "precision": 0},
        # the same work in the mixed-precision form
        {"name": "adapt3d_mixed_40", "kind": "adapt", "dim": 3, "n": 40, "metric": "levelset",
         "elems": 0, "aspect": 1.0, "precision": 1},
        # a simulation's remesh: an isotropic metric and the solution's fields
        {"name": "adapt3d_tags", "kind": "tags", "dim": 3, "n": 14, "metric": "sphere",
         "elems": 0, "aspect": 1.0, "precision": 0},
        # many small meshes adapted in one call
        {"name": "batch_small", "kind": "batch", "dim": 3, "n": 6, "count": 16, "elems": 2000,
         "aspect": 1.5},
        # lengths and qualities of a large mesh on device arrays
        {"name": "measure_80", "kind": "measure", "dim": 3, "n": 80},
        # metric preparation: the mesh's implied metrics, and gradation limiting of a
        # size field with a sharp jump
        {"name": "metric_31", "kind": "metric", "dim": 3, "n": 31, "rate": 0.5},
        # building the input mesh
        {"name": "build_40", "kind": "build", "dim": 3, "n": 40},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("level", "level", "constant3", "constant2", "ring", "tags", "batch",
                       "measure", "metric", "build"))
    if kind == "level":
        return {"kind": "adapt", "dim": 3, "n": _log_int(rng, 5, 56), "metric": "levelset",
                "elems": 0, "aspect": 1.0, "precision": int(rng.random() < 0.25)}
    if kind == "constant3":
        return {"kind": "adapt", "dim": 3, "n": _log_int(rng, 3, 20), "metric": "constant",
                "elems": _log_int(rng, 300, 30000), "aspect": round(rng.uniform(1.2, 2.0), 2),
                "precision": 0}
    if kind == "constant2":
        return {"kind": "adapt", "dim": 2, "n": _log_int(rng, 4, 120), "metric": "constant",
                "elems": _log_int(rng, 300, 60000), "aspect": round(rng.uniform(1.2, 4.0), 2),
                "precision": 0}
    if kind == "ring":
        return {"kind": "adapt", "dim": 2, "n": _log_int(rng, 8, 200), "metric": "ring",
                "elems": 0, "aspect": 1.0, "precision": 0}
    if kind == "tags":
        return {"kind": "tags", "dim": 3, "n": _log_int(rng, 4, 16), "metric": "sphere",
                "elems": 0, "aspect": 1.0, "precision": 0}
    if kind == "batch":
        return {"kind": "batch", "dim": 3, "n": _log_int(rng, 3, 8),
                "count": _log_int(rng, 4, 16), "elems": _log_int(rng, 300, 3000),
                "aspect": round(rng.uniform(1.2, 1.8), 2)}
    if kind == "measure":
        return {"kind": "measure", "dim": rng.choice((2, 3)), "n": _log_int(rng, 8, 80)}
    if kind == "metric":
        return {"kind": "metric", "dim": rng.choice((2, 3)), "n": _log_int(rng, 6, 31),
                "rate": round(rng.uniform(0.3, 1.0), 2)}
    return {"kind": "build", "dim": rng.choice((2, 3)), "n": _log_int(rng, 5, 40)}


# ------------------------------------------------------------------ inputs


def _rotation(dim, rng):
    q, r = np.linalg.qr(rng.normal(size=(dim, dim)))
    return q * np.sign(np.diag(r))


def _components(m, dim):
    if dim == 3:
        return np.array([m[0, 0], m[1, 1], m[2, 2], m[0, 1], m[1, 2], m[0, 2]])
    return np.array([m[0, 0], m[1, 1], m[0, 1]])


def _constant(dim, elems, aspect, rng):
    """A constant metric for about `elems` elements in the unit box: random
    axes, neighbouring eigen-lengths `aspect` apart."""
    lam = aspect ** (2.0 * np.arange(dim))
    q = _rotation(dim, rng)
    v = _components(q @ np.diag(lam) @ q.T, dim)
    return v * (elems / W.expected_nelems_unit_box(v, dim)) ** (2.0 / dim)


def _sphere_metric(coords, rng):
    """Isotropic sizes growing away from a sphere whose centre is drawn."""
    p = coords.reshape(-1, 3)
    c = 0.5 + rng.uniform(-0.05, 0.05, 3)
    h = 0.07 + 0.25 * np.abs(np.linalg.norm(p - c, axis=1) - 0.3)
    return 1.0 / (h * h), 1


def _metric(case, coords, rng):
    dim = case["dim"]
    if case["metric"] == "ring":
        return W.iso_ring_metric_2d(coords + rng.uniform(-0.05, 0.05))
    if case["metric"] == "levelset":
        return W.levelset_metric_3d(coords, amplitude=rng.uniform(0.095, 0.105))
    if case["metric"] == "sphere":
        return _sphere_metric(coords, rng)
    v = _constant(dim, case["elems"], case["aspect"], rng)
    return np.tile(v, coords.size // dim), len(v)


def _opts(dim, precision=0):
    o = _context().default_opts(dim)
    o.verbosity = 0
    o.precision = precision
    return o


def _box(case, rng):
    """The input mesh with its metric, as adapt() gets it."""
    m = A.Mesh.box(_context(), case["dim"], case["n"])
    metric, ncomps = _metric(case, m.coords(), rng)
    m.set_metric(metric, ncomps)
    return m


def _jittered(case, rng):
    """A box whose vertices are moved a little, as a mesh that has moved is."""
    dim, n = case["dim"], case["n"]
    m = A.Mesh.box(_context(), dim, n)
    x = m.coords()
    m.set_coords(x + rng.uniform(-0.15 / n, 0.15 / n, x.size))
    return m


def _jump(m, n, rng):
    """Isotropic sizes eight times smaller inside a sphere than outside."""
    p = m.coords().reshape(m.nents(0), -1)
    c = 0.5 + rng.uniform(-0.1, 0.1, p.shape[1])
    h = np.where(np.linalg.norm(p - c, axis=1) < 0.25, 0.5 / n, 4.0 / n)
    return 1.0 / (h * h)


# more entities than a case's adapted mesh has: its result goes into buffers
# of this size, which a program keeps
def _capacity(case):
    metric = case.get("metric", "constant")
    if metric == "constant":
        return 4 * case["elems"] + 2000
    return {"ring": 20000, "levelset": 400000, "sphere": 60000}[metric]


def _buffers(case):
    dim, cap = case["dim"], _capacity(case)
    nc = 1 if case.get("metric") in ("ring", "sphere") else (6 if dim == 3 else 3)

    def full(k, dtype):
        return torch.full((k,), -1, dtype=dtype, device="cuda")

    return {"verts": full(cap * (dim + 1), torch.int32),
            "coords": full(cap * dim, torch.float64), "metric": full(cap * nc, torch.float64)}


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind, dim = case["kind"], case["dim"]
    s = {"case": case}
    if kind == "adapt":
        s["mesh"] = _box(case, rng)
        s["opts"] = _opts(dim, case["precision"])
        s["out"] = _buffers(case)
    elif kind == "tags":
        m = _box(case, rng)
        x = m.coords().reshape(-1, dim)
        v = m.verts(dim).reshape(-1, dim + 1)
        xc = x[v].mean(axis=1)
        w = rng.uniform(1.0, 3.0, dim)
        m.add_vertex_tag("temperature", 1, A.Mesh.LINEAR, np.sin(x @ w))
        m.add_elem_tag("material", 1, np.floor(4.0 * xc[:, 0]))
        m.add_elem_tag("density", 1, 1.0 + 0.5 * np.cos(xc @ w))
        m.set_elem_transfer("density", A.Mesh.CONSERVE)
        s["mesh"], s["opts"], s["out"] = m, _opts(dim), _buffers(case)
        for name in ("temperature", "material", "density"):
            s["out"][name] = torch.full((_capacity(case),), -1, dtype=torch.float64,
                                        device="cuda")
    elif kind == "batch":
        s["meshes"] = []
        for k in range(case["count"]):
            one = dict(case, n=max(2, case["n"] - k % 3), metric="constant")
            s["meshes"].append(_box(one, rng))
        s["opts"] = _opts(dim)
        s["out"] = [_buffers(case) for _ in s["meshes"]]
    elif kind == "measure":
        m = _jittered(case, rng)
        m.set_metric(*W.banded_aniso_metric(m.coords(), dim, rng))
        s["ncomps"] = m.metric_ncomps
        s["elems"] = _cuda(m.verts(dim))
        s["edges"] = _cuda(m.verts(1))
        s["coords"] = _cuda(m.coords())
        s["metric"] = _cuda(m.metric())
        s["quality"] = torch.empty(m.nents(dim), dtype=torch.float64, device="cuda")
        s["length"] = torch.empty(m.nents(1), dtype=torch.float64, device="cuda")
    elif kind == "metric":
        s["mesh"] = _jittered(case, rng)
        s["sizes"] = _cuda(_jump(s["mesh"], case["n"], rng))
    else:
        s["size"] = [float(v) for v in rng.uniform(0.5, 2.0, dim)]
    return s


# ------------------------------------------------------------------ passes


def _pointer(t, ctype):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctype))


def _reals(n):
    return torch.empty(n, dtype=torch.float64, device="cuda")


def _result(m, out):
    """The mesh as a program on the GPU takes it: element vertices,
    coordinates and metric, at the start of the program's buffers."""
    dim, nv = m.dim, m.nents(0)
    for name, n in (("verts", m.nents(dim) * (dim + 1)), ("coords", nv * dim),
                    ("metric", nv * m.metric_ncomps)):
        if n > out[name].numel():
            raise RuntimeError("the adapted mesh does not fit the buffers")
    A.check(m.lib.osh_mesh_get_verts(m.h, dim, _pointer(out["verts"], ctypes.c_int)), m.lib)
    A.check(m.lib.osh_mesh_get_coords(m.h, _pointer(out["coords"], ctypes.c_double)), m.lib)
    A.check(m.lib.osh_mesh_get_metric(m.h, _pointer(out["metric"], ctypes.c_double)), m.lib)
    return dict(out, elems=m.nents(dim), nverts=nv)


def _run_adapt(s):
    m = s["mesh"].copy()
    did, passes = m.adapt(s["opts"])
    return m, dict(_result(m, s["out"]), did=did, passes=len(passes))


def run(s):
    kind, dim = s["case"]["kind"], s["case"]["dim"]
    if kind == "adapt":
        return _run_adapt(s)[1]
    if kind == "tags":
        m, out = _run_adapt(s)
        for name, getter in (("temperature", m.lib.osh_mesh_get_vertex_tag),
                             ("material", m.lib.osh_mesh_get_elem_tag),
                             ("density", m.lib.osh_mesh_get_elem_tag)):
            A.check(getter(m.h, name.encode(), _pointer(out[name], ctypes.c_double)), m.lib)
        return out
    if kind == "batch":
        meshes = [m.copy() for m in s["meshes"]]
        did, _, _ = A.adapt_batch(meshes, s["opts"])
        # at most 64 arrays: the meshes' counts in one list of their own
        got = [_result(m, out) for m, out in zip(meshes, s["out"])]
        return {"meshes": [[r["verts"], r["coords"], r["metric"]] for r in got],
                "counts": np.array([[r["elems"], r["nverts"]] for r in got] +
                                   [[d, 0] for d in did])}
    ctx = _context()
    if kind == "measure":
        x, metric = s["coords"].data_ptr(), s["metric"].data_ptr()
        ctx.measure_qualities(dim, s["ncomps"], s["quality"].numel(), s["elems"].data_ptr(), x,
                              metric, s["quality"].data_ptr())
        ctx.measure_edges_metric(dim, s["ncomps"], s["length"].numel(), s["edges"].data_ptr(), x,
                                 metric, s["length"].data_ptr())
        return {"quality": s["quality"], "length": s["length"]}
    if kind == "metric":
        m = s["mesh"].copy()
        implied = _reals(m.nents(0) * dim * (dim + 1) // 2)
        graded = _reals(m.nents(0))
        A.check(m.lib.osh_get_implied_metrics(m.h, 0, _pointer(implied, ctypes.c_double)), m.lib)
        A.check(m.lib.osh_mesh_set_metric(m.h, 1, _pointer(s["sizes"], ctypes.c_double)), m.lib)
        sweeps = m.limit_metric_gradation(s["case"]["rate"])
        A.check(m.lib.osh_mesh_get_metric(m.h, _pointer(graded, ctypes.c_double)), m.lib)
        return {"implied": implied, "graded": graded, "sweeps": sweeps}
    x, y = s["size"][:2]
    m = A.Mesh.box(ctx, dim, s["case"]["n"], x=x, y=y, z=s["size"][2] if dim == 3 else 1.0)
    out = {}
    for d in range(1, dim + 1):
        t = torch.empty(m.nents(d) * (d + 1), dtype=torch.int32, device="cuda")
        A.check(m.lib.osh_mesh_get_verts(m.h, d, _pointer(t, ctypes.c_int)), m.lib)
        out["verts%d" % d] = t
    out["coords"] = _reals(m.nents(0) * dim)
    A.check(m.lib.osh_mesh_get_coords(m.h, _pointer(out["coords"], ctypes.c_double)), m.lib)
    return out


# ------------------------------------------------------- work and tolerance


def _counts(dim, n):
    """Vertices, edges and elements of an n-cells-per-side box."""
    nv = (n + 1) ** dim
    if dim == 2:
        return nv, 3 * n * n + 2 * n, 2 * n * n
    return nv, 7 * n ** 3 + 9 * n * n + 3 * n, 6 * n ** 3


def work(case):
    """Each input and output array once.  An adapted mesh is taken to have
    the expected number of elements of a constant metric, else as many as went
    in."""
    kind, dim, n = case["kind"], case["dim"], case["n"]
    nv, ne, nt = _counts(dim, n)
    if kind == "measure":
        nc = 6 if dim == 3 else 3
        flops = (222 * nt + 60 * ne) if dim == 3 else (80 * nt + 40 * ne)
        return {"bytes": nv * 2 * 8 * (dim + nc) + nt * (4 * (dim + 1) + 8) + ne * 16,
                "flops": flops}
    if kind == "metric":
        nc = 6 if dim == 3 else 3
        return {"bytes": nv * 8 * (dim + nc + 2) + nt * 4 * (dim + 1), "flops": 0}
    if kind == "build":
        nf = 12 * n ** 3 + 6 * n * n if dim == 3 else 0
        return {"bytes": nv * 8 * dim + ne * 8 + nf * 12 + nt * 4 * (dim + 1), "flops": 0}
    nc = 1 if case.get("metric") in ("ring", "sphere") else (6 if dim == 3 else 3)
    vert, elem = 8 * (dim + nc), 4 * (dim + 1)
    out = case["elems"] or nt
    bytes_ = nv * vert + nt * elem + (out / nt) * nv * vert + out * elem
    return {"bytes": bytes_ * case.get("count", 1), "flops": 0}


def tolerance(case):
    """A rebuilt mesh is a chain of decisions, each on values that are the
    same bit for bit in every form of the framework, so meshes and what they
    carry are compared exactly.  Measures and metrics are formulas in 64 bits;
    the rates are four times what the plain formulas in exact() differ by."""
    if case["kind"] == "measure":
        return {"rel": 1.2e-14, "max": 1e-11}
    if case["kind"] == "metric":
        return {"rel": 4e-10, "max": 4e-8}
    return "exact"


# ---------------------------------------------------------------- reference


def _symmetric(v, dim):
    """Stored components to matrices."""
    i = [[0, 3, 5], [3, 1, 4], [5, 4, 2]] if dim == 3 else [[0, 2], [2, 1]]
    return v[..., torch.tensor(i, device=v.device)]


def _exact_measures(s, dim):
    x = s["coords"].reshape(-1, dim)
    m = _symmetric(s["metric"].reshape(x.shape[0], -1), dim)
    ev = s["edges"].reshape(-1, 2).long()
    d = x[ev[:, 1]] - x[ev[:, 0]]

    def norm2(mat, vec):
        return (vec * (mat * vec[:, None, :]).sum(-1)).sum(-1)

    a, b = norm2(m[ev[:, 0]], d).sqrt(), norm2(m[ev[:, 1]], d).sqrt()
    length = torch.where((a - b).abs() > 1e-3, (a - b) / torch.log(a / b), (a + b) / 2)
    tv = s["elems"].reshape(-1, dim + 1).long()
    det = torch.linalg.det(m.cpu()).to(x.device)
    best = det[tv].argmax(dim=1)
    top = torch.gather(tv, 1, best[:, None])[:, 0]
    p = x[tv]
    basis = p[:, 1:] - p[:, :1]
    if dim == 3:
        size = (torch.linalg.cross(basis[:, 0], basis[:, 1]) * basis[:, 2]).sum(-1) / 6.0
        equilateral = 0.1178511301977579
    else:
        size = (basis[:, 0, 0] * basis[:, 1, 1] - basis[:, 0, 1] * basis[:, 1, 0]) / 2.0
        equilateral = 0.4330127018922193
    size = size * det[top].sqrt()
    pairs = [(i, j) for i in range(dim + 1) for j in range(i)]
    mean = sum(norm2(m[top], p[:, i] - p[:, j]) for i, j in pairs) / len(pairs)
    ratio = (size / equilateral).abs()
    quality = torch.where(size < 0, size, (ratio ** (2.0 / 3.0) if dim == 3 else ratio) / mean)
    return {"quality": quality, "length": length}


def _exact_implied(m, dim):
    """The log-Euclidean mean over each vertex's elements of the metric in
    which every edge of the element has unit length, scaled to a typical
    element's size."""
    x = m.coords().reshape(-1, dim)
    tv = m.verts(dim).reshape(-1, dim + 1)
    d = np.stack([x[tv[:, j]] - x[tv[:, i]] for i in range(dim + 1)
                  for j in range(i + 1, dim + 1)], axis=1)
    off = [(0, 1), (1, 2), (0, 2)] if dim == 3 else [(0, 1)]
    rows = np.concatenate([d * d, np.stack([2 * d[..., i] * d[..., j] for i, j in off], -1)], -1)
    comps = np.linalg.solve(rows, np.ones(rows.shape[:2] + (1,)))[..., 0]
    typical, perfect = (0.0838934100219, 0.1178511301977579) if dim == 3 else \
        (0.377645136635, 0.4330127018922193)
    comps = comps * (typical / perfect) ** (2.0 / dim)

    def spectral(v, f):
        w, q = np.linalg.eigh(_symmetric(torch.from_numpy(v), dim).numpy())
        mat = (q * f(w)[:, None, :]) @ q.transpose(0, 2, 1)
        return np.stack([mat[:, i, i] for i in range(dim)] + [mat[:, i, j] for i, j in off], -1)

    logs = spectral(comps, np.log)
    out = np.zeros((len(x), comps.shape[1]))
    count = np.zeros(len(x))
    for k in range(dim + 1):
        np.add.at(out, tv[:, k], logs)
        np.add.at(count, tv[:, k], 1.0)
    return spectral(out / count[:, None], np.exp).ravel()


def _exact_graded(s, dim, rate):
    """Sweeps of m(v) = max(m(v), m(u) / (1 + rate d_u(u, v))^2) over the
    edges until no value moves by more than 1 %."""
    x = s["mesh"].coords().reshape(-1, dim)
    ev = s["mesh"].verts(1).reshape(-1, 2)
    dist = np.linalg.norm(x[ev[:, 1]] - x[ev[:, 0]], axis=1)
    m = s["sizes"].cpu().numpy()
    while True:
        out = m.copy()
        for a, b in ((0, 1), (1, 0)):
            near = m[ev[:, b]]
            np.maximum.at(out, ev[:, a], near / (1.0 + np.sqrt(near) * dist * rate) ** 2)
        if np.all(np.abs(out - m) / np.maximum(out, m) <= 1e-2):
            return out
        m = out


def exact(case, seed):
    """The formulas in plain torch and numpy.  An adapted mesh and a built
    numbering have no such value."""
    if case["kind"] == "measure":
        return _exact_measures(prepare(case, seed), case["dim"])
    if case["kind"] == "metric":
        s = prepare(case, seed)
        return {"implied": torch.from_numpy(_exact_implied(s["mesh"], case["dim"])),
                "graded": torch.from_numpy(_exact_graded(s, case["dim"], case["rate"])),
                "sweeps": None}
    return None
