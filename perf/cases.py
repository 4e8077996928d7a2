"""The work a user of this framework has it do, as cases that can be timed.

Eight kinds of pass, each through the public entry points of ``nosh_amd``:

operators     F(psi), K phi and J(psi) phi on device vectors: what an outer
              Newton-Krylov library calls between its own vector updates
minres        one preconditioned linear solve, host vectors in and out
newton        Newton steps with a fixed inner budget on a device vector, in
              FP64 throughout or with the FP32 inner solver
continuation  a whole natural-parameter continuation with the tangent predictor
batch         lockstep Newton steps of many branches on one or more meshes
train, infer  the surrogate network: Adam steps on minibatches, inference
eigen         the stability eigenvalues of a converged state
mesh          the edge/covolume cache of a new mesh

Inner solves run a fixed number of iterations, so that what a pass computes
does not hang on a tolerance met one iteration earlier or later. Meshes are
Kuhn boxes and split squares on [-5, 5], the magnetic field is constant along
z, V = -1, unit thickness.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import nosh_amd as nosh

DEV = "cuda" if torch.cuda.is_available() else "cpu"
CHEB, RATIO = 6, 300.0


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # The smallest meshes of the tests: a pass is launches and nothing else.
        dict(name="operators square 16", kind="operators", dim=2, nx=16, ny=16, nz=0, jitter=0.0),
        # The benchmark's mesh: every apply streams the whole matrix.
        dict(name="operators cube 96", kind="operators", dim=3, nx=96, ny=96, nz=96, jitter=0.0),
        # A linear solve at the size of the reference's own 2D examples, with
        # host vectors as a Trilinos caller has them.
        dict(name="minres square 61x67", kind="minres", dim=2, nx=61, ny=67, nz=0, jitter=0.0,
             iters=48),
        # The plain solver on the benchmark's mesh.
        dict(name="newton fp64 cube 96", kind="newton", dim=3, nx=96, ny=96, nz=96, jitter=0.0,
             precision=0, steps=1, iters=24),
        # The mixed-precision solver on a mesh of ordinary size, nothing round.
        dict(name="newton mixed box 53x41x47", kind="newton", dim=3, nx=53, ny=41, nz=47,
             jitter=0.2, precision=1, steps=2, iters=16),
        # A whole run of the single-branch driver in 2D.
        dict(name="continuation square 64", kind="continuation", dim=2, nx=64, ny=64, nz=0,
             jitter=0.0, steps=4),
        # The benchmark's batch: eight branches on its mesh, at one mu, with
        # the tuning its autotuner picks there.
        dict(name="batch cube 96 x 8", kind="batch", nx=96, ny=96, nz=96, jitter=0.0, groups=1,
             lanes=8, shared_mu=True, steps=2, iters=16, threads=512, fold=8, mode=2),
        # A batch of random instances over meshes of uneven size, every
        # instance at a mu of its own, as it is created.
        dict(name="batch three boxes x 7", kind="batch", nx=17, ny=21, nz=19, jitter=0.2,
             groups=3, lanes=7, shared_mu=False, steps=2, iters=16, threads=256, fold=1, mode=0),
        # One burst of surrogate training at the default minibatch.
        dict(name="train 16384", kind="train", rows=16384, width=256, depth=4, steps=4),
        # The surrogate's guess for one branch on the benchmark's mesh.
        dict(name="infer 912673", kind="infer", rows=912673, width=256, depth=4),
        # Stability of a converged 2D state.
        dict(name="eigen square 32", kind="eigen", dim=2, nx=32, ny=32, nz=0, jitter=0.0, nev=4),
        # A program's first call on a new mesh.
        dict(name="mesh box 47x53x43", kind="mesh", dim=3, nx=47, ny=53, nz=43, jitter=0.2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["operators", "minres", "newton", "continuation", "batch", "batch", "train",
                       "infer", "eigen", "mesh"])
    if kind == "train":
        return dict(kind=kind, rows=_log(rng, 500, 16384), width=rng.choice([64, 128, 256]),
                    depth=rng.randint(2, 4), steps=rng.randint(1, 4))
    if kind == "infer":
        return dict(kind=kind, rows=_log(rng, 1000, 900000), width=rng.choice([64, 128, 256]),
                    depth=rng.randint(2, 4))
    if kind == "continuation":
        n = _log(rng, 16, 64)
        return dict(kind=kind, dim=2, nx=n, ny=n, nz=0, jitter=0.0, steps=rng.randint(2, 4))
    if kind == "eigen":
        n = _log(rng, 12, 32)
        return dict(kind=kind, dim=2, nx=n, ny=n, nz=0, jitter=0.0, nev=rng.randint(1, 4))
    if kind == "batch":
        lanes, groups = rng.randint(2, 12), rng.randint(1, 3)
        n = _log(rng, 8, min(64, int(97 * (8 / (16 * groups)) ** (1 / 3))))
        mode = rng.choice([0, 2])
        return dict(kind=kind, nx=n, ny=n + rng.randint(0, 3), nz=max(4, n - rng.randint(0, 3)),
                    jitter=rng.choice([0.0, 0.2]), groups=groups, lanes=lanes,
                    shared_mu=rng.random() < 0.5, steps=2, iters=rng.randint(8, 16),
                    threads=rng.choice([256, 512]), fold=rng.choice([1, 4, 8]), mode=mode)
    dim = rng.choice([2, 3, 3])
    if dim == 2:
        nx, ny, nz = _log(rng, 12, 400), _log(rng, 12, 400), 0
    else:
        top = 47 if kind == "mesh" else 88
        n = _log(rng, 6, top)
        nx, ny, nz = n, n + rng.randint(0, 5), max(5, n - rng.randint(0, 5))
    moved = kind == "mesh" or (dim == 3 and rng.random() < 0.6)
    case = dict(kind=kind, dim=dim, nx=nx, ny=ny, nz=nz, jitter=0.2 if moved else 0.0)
    if kind == "minres":
        case.update(iters=rng.randint(8, 24) if dim == 3 else rng.randint(16, 48))
    if kind == "newton":
        precision = rng.randint(0, 1)
        case.update(precision=precision, steps=1 + precision, iters=rng.randint(8, 16))
    return case


# ------------------------------------------------------------------ the meshes
def _grid(dim, nx, ny, nz):
    """Vertices of a box (or rectangle), its longest side spanning [-5, 5]."""
    h = 10.0 / max(nx, ny, nz)
    ax = [(np.arange(k + 1) - 0.5 * k) * h for k in ((nx, ny, nz) if dim == 3 else (nx, ny))]
    mesh = np.meshgrid(*reversed(ax), indexing="ij")
    xyz = np.zeros((mesh[0].size, 3))
    for d, a in enumerate(reversed(mesh)):
        xyz[:, d] = a.ravel()
    return xyz, h


def _cells(dim, nx, ny, nz):
    """Two triangles a square, or the six Kuhn tetrahedra of a cube."""
    if dim == 2:
        b = (np.arange(ny)[:, None] * (nx + 1) + np.arange(nx)[None, :]).ravel()
        s = (1, nx + 1)
        t = [(b, b + s[0], b + s[0] + s[1]), (b, b + s[0] + s[1], b + s[1])]
    else:
        s = (1, nx + 1, (nx + 1) * (ny + 1))
        b = (np.arange(nz)[:, None, None] * s[2] + np.arange(ny)[None, :, None] * s[1]
             + np.arange(nx)[None, None, :]).ravel()
        orders = ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))
        t = [(b, b + s[i], b + s[i] + s[j], b + sum(s)) for i, j, _ in orders]
    out = np.empty((len(t) * b.size, dim + 1), dtype=np.int32)
    for k, c in enumerate(t):
        out[k::len(t)] = np.stack(c, axis=1)
    return out


def _box(dim, nx, ny, nz, jitter, seed):
    xyz, h = _grid(dim, nx, ny, nz)
    if jitter > 0.0:  # interior vertices moved by up to jitter h
        top = xyz.max(axis=0)
        inner = np.all(np.abs(xyz[:, :dim]) < top[:dim] - 0.5 * h, axis=1)
        rng = np.random.default_rng(seed)
        xyz[inner, :dim] += rng.uniform(-jitter * h, jitter * h, (int(inner.sum()), dim))
    return xyz, _cells(dim, nx, ny, nz)


def _potential(xyz):
    return np.stack([-0.5 * xyz[:, 1], 0.5 * xyz[:, 0], np.zeros(len(xyz))], axis=1)


def _boxes(case):
    """The boxes (dim, nx, ny, nz, jitter) of a case, one per mesh."""
    if case["kind"] == "batch":
        return [(3, case["nx"] + 4 * k, case["ny"] + k, case["nz"] + 2 * k, case["jitter"])
                for k in range(case["groups"])]
    return [(case["dim"], case["nx"], case["ny"], case["nz"], case["jitter"])]


@functools.lru_cache(maxsize=4)
def _mesh(box):
    """A program builds its mesh once and solves on it many times."""
    xyz, cells = _box(*box, seed=2)
    return nosh.Mesh(xyz, cells), _potential(xyz)


def _model(box, mu, g):
    mesh, A = _mesh(box)
    mvp = nosh.VectorFieldExplicitValues(mesh, A, mu)
    V = nosh.ScalarFieldConstant(mesh, -1.0)
    t = nosh.ScalarFieldConstant(mesh, 1.0)
    return mesh, nosh.Nls(mesh, mvp, V, g, t), nosh.Keo(mesh, t, mvp)


def _vertices(box):
    dim, nx, ny, nz, _ = box
    return (nx + 1) * (ny + 1) * (nz + 1 if dim == 3 else 1)


def _edges(box):
    dim, nx, ny, nz, _ = box
    if dim == 2:
        return nx * (ny + 1) + ny * (nx + 1) + nx * ny
    axes = (nx * (ny + 1) * (nz + 1) + ny * (nx + 1) * (nz + 1) + nz * (nx + 1) * (ny + 1))
    faces = nx * ny * (nz + 1) + nx * nz * (ny + 1) + ny * nz * (nx + 1)
    return axes + faces + nx * ny * nz


# ------------------------------------------------------------------ the inputs
def _parameters(case, seed):
    """mu and g of every instance: a Meissner state's range."""
    rng = np.random.default_rng([seed, 1])
    count = case.get("groups", 1) * case.get("lanes", 1)
    g = rng.uniform(0.6, 2.0, count)
    mu = rng.uniform(0.02, 0.08, count)
    if case.get("shared_mu", True):
        mu[:] = mu[0]
    return mu, g


def _random(n, seed, what):
    """A state with moduli in [0.5, 1] and any phase."""
    rng = np.random.default_rng([seed, 2, what])
    z = rng.uniform(0.5, 1.0, n) * np.exp(2j * np.pi * rng.random(n))
    return z.view(np.float64)


def _near(n, g, seed, what):
    """A guess near the superconducting state, as a predictor leaves it."""
    rng = np.random.default_rng([seed, 3, what])
    z = (1.0 + 0.01 * rng.standard_normal(n)) * np.exp(0.01j * rng.standard_normal(n))
    return (z / math.sqrt(g)).view(np.float64)


def _network(case, seed):
    """Weights (BF16 values, layer by layer, each [out][in]) and biases."""
    gen = torch.Generator().manual_seed(seed * 7 + 5)
    dims = [7] + [case["width"]] * case["depth"] + [2]
    w, b = [], []
    for i, o in zip(dims, dims[1:]):
        a = math.sqrt(6.0 / i) * (0.1 if o == 2 else 1.0)
        w.append(((2 * torch.rand(o, i, generator=gen) - 1) * a).bfloat16().float())
        b.append(0.1 * (2 * torch.rand(o, generator=gen) - 1))
    return w, b


def _samples(rows, seed, what):
    gen = torch.Generator(device=DEV).manual_seed(seed * 13 + what)
    x = 2 * torch.rand(rows, 7, generator=gen, device=DEV) - 1
    y = torch.stack([torch.sin(2 * x[:, 0]) * x[:, 3], x[:, 1] * x[:, 4] - 0.5 * x[:, 6]], 1)
    return x, y.contiguous()


def _mlp(case, seed):
    net = nosh.Mlp(n_in=7, width=case["width"], depth=case["depth"], n_out=2, seed=0)
    w, b = _network(case, seed)
    net.set_params(torch.cat([t.ravel() for t in w] + b).numpy())
    return net


# --------------------------------------------------------------- prepare, run
def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "train":
        s.update(net=_mlp(case, seed),
                 data=[_samples(case["rows"], seed, k) for k in range(case["steps"])])
    elif kind == "infer":
        x, _ = _samples(case["rows"], seed, 0)
        s.update(net=_mlp(case, seed), x=x, y=torch.empty(case["rows"], 2, device=DEV))
    elif kind == "mesh":
        s["xyz"], s["cells"] = _box(*_boxes(case)[0], seed=seed)
    else:
        mu, g = _parameters(case, seed)
        boxes = _boxes(case)
        if kind == "batch":
            lanes = case["lanes"]
            s["models"] = [_model(b, mu[k * lanes], g[k * lanes])[1] for k, b in enumerate(boxes)]
            s["batch"] = nosh.Batch([(m, lanes) for m in s["models"]], mu, g)
            s["batch"].set_tuning(case["threads"], case["mode"], 4, 16, fold=case["fold"])
            s["start"] = torch.from_numpy(np.concatenate(
                [_near(_vertices(b), g[k * lanes + i], seed, k * lanes + i)
                 for k, b in enumerate(boxes) for i in range(lanes)])).to(DEV)
            s["psi"] = torch.empty_like(s["start"])
        else:
            _prepare_single(s, case, seed, boxes[0], float(mu[0]), float(g[0]))
    if DEV == "cuda":
        torch.cuda.synchronize()
    return s


def _prepare_single(s, case, seed, box, mu, g):
    kind, n = case["kind"], _vertices(box)
    s["params"] = p = {"g": g, "mu": mu}
    s["mesh"], s["model"], keo = _model(box, mu, g)
    if kind == "operators":
        psi = _random(n, seed, 0)
        s["psi"] = torch.from_numpy(psi).to(DEV)
        s["phi"] = torch.from_numpy(_random(n, seed, 1)).to(DEV)
        s["keo"], s["jac"] = keo, s["model"].create_W_op()
        keo.set_parameters(p)
        s["jac"].rebuild(p, psi)
        for k in ("psi_in", "f_in", "f", "kphi", "jphi"):
            s[k] = torch.empty_like(s["psi"])
    elif kind == "minres":
        psi = _near(n, g, seed, 0)
        s["b"] = s["model"].eval_f(psi, p)
        s["jac"], s["prec"] = s["model"].create_W_op(), s["model"].create_W_prec()
        s["prec"].set_chebyshev(CHEB, RATIO)
        s["jac"].rebuild(p, psi)
        s["prec"].rebuild(p, psi)
    elif kind == "newton":
        s["start"] = torch.from_numpy(_near(n, g, seed, 0)).to(DEV)
        s["psi"] = torch.empty_like(s["start"])
    elif kind == "continuation":
        s["psi0"] = np.full(n, 1.0 / math.sqrt(g), dtype=np.complex128).view(np.float64)
        s["stop"] = 0.1 + mu
    elif kind == "eigen":
        s["params"] = p = {"g": g, "mu": 0.1 + mu}
        psi = np.full(n, 1.0 / math.sqrt(g), dtype=np.complex128).view(np.float64)
        s["psi"], _ = nosh.newton_solve(s["model"], psi, p, tol=1e-11)


def _phase_fixed(z):
    """The state with its mean real and positive: solutions come with any
    global phase, and a program that keeps or compares them fixes it."""
    m = z.mean()
    return (z * (m.conjugate() / abs(m))).view(np.float64)


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "operators":
        s["mesh"].to_internal(s["psi"].data_ptr(), s["psi_in"].data_ptr())
        s["model"].eval_f_internal(s["psi_in"].data_ptr(), s["params"], s["f_in"].data_ptr())
        s["mesh"].to_reference(s["f_in"].data_ptr(), s["f"].data_ptr())
        s["keo"].apply_device(s["phi"].data_ptr(), s["kphi"].data_ptr())
        s["jac"].apply_device(s["phi"].data_ptr(), s["jphi"].data_ptr())
        return s["f"], s["kphi"], s["jphi"]
    if kind == "minres":
        x, _, _ = nosh.minres_solve(s["jac"], s["prec"], s["b"], rtol=0.0,
                                    max_iters=case["iters"])
        return x
    if kind == "newton":
        s["psi"].copy_(s["start"])
        torch.cuda.current_stream().synchronize()
        nosh.newton_solve_device(s["model"], s["psi"].data_ptr(), s["params"], tol=0.0,
                                 max_iters=case["steps"], minres_rtol=0.0,
                                 minres_max_iters=case["iters"], cheb_iters=CHEB,
                                 cheb_ratio=RATIO, precision=case["precision"])
        return s["psi"]
    if kind == "continuation":
        psi, rec = nosh.continuation(s["model"], s["psi0"], s["params"], "mu", 0.0, s["stop"],
                                     case["steps"], tol=1e-12, cheb_iters=CHEB,
                                     cheb_ratio=RATIO)
        return _phase_fixed(psi.view(np.complex128)), [r["gibbs"] for r in rec]
    if kind == "batch":
        s["psi"].copy_(s["start"])
        torch.cuda.current_stream().synchronize()
        s["batch"].solve_device(s["psi"].data_ptr(), tol=0.0, max_iters=case["steps"],
                                minres_rtol=0.0, minres_max_iters=case["iters"], cheb_iters=5,
                                cheb_ratio=RATIO)
        return s["psi"]
    if kind == "train":
        for x, y in s["data"]:
            s["net"].train_step_device(x.data_ptr(), y.data_ptr(), case["rows"], 1e-4)
        return s["net"].get_params()
    if kind == "infer":
        s["net"].infer_device(s["x"].data_ptr(), case["rows"], s["y"].data_ptr())
        return s["y"]
    if kind == "eigen":
        ev, _, _ = nosh.jacobian_eigenpairs(s["model"], s["psi"], s["params"], nev=case["nev"],
                                          tol=1e-9)
        return ev
    mesh = nosh.Mesh(s["xyz"], s["cells"])
    length, covolume = mesh.get_edge_data()
    return mesh.my_edges(), length, covolume, mesh.control_volumes()


# ------------------------------------------------------------------------ work
def work(case):
    """What one pass cannot do without. A product with K, J or P reads every
    edge's complex value and its two vertex numbers once and every row's
    entries once (8 real operations an edge and direction)."""
    kind = case["kind"]
    if kind in ("train", "infer"):
        w, d, m = case["width"], case["depth"], case["rows"]
        weights = 7 * w + (d - 1) * w * w + 2 * w
        if kind == "infer":
            return {"bytes": 4.0 * m * 9 + 2.0 * weights, "flops": 2.0 * m * weights}
        return {"bytes": case["steps"] * (4.0 * m * 9 + 28.0 * weights),
                "flops": case["steps"] * 6.0 * m * weights}
    nbytes = flops = 0.0
    for box in _boxes(case):
        n, e = _vertices(box), _edges(box)
        if kind == "mesh":
            cells = (6 * case["nx"] * case["ny"] * case["nz"] if case["dim"] == 3
                     else 2 * case["nx"] * case["ny"])
            nbytes += 24.0 * n + 4.0 * (case["dim"] + 1) * cells + 24.0 * e + 8.0 * n
            flops += 300.0 * cells
            continue
        value, entry = 24.0, 16.0  # an edge's value and numbers; a complex entry
        if kind == "newton" and case["precision"] == 1:
            value, entry = 16.0, 8.0
        apply_b, apply_f = value * e + 3.5 * entry * n, 16.0 * e + 14.0 * n
        if kind == "operators":
            nbytes += 3.0 * apply_b
            flops += 3.0 * apply_f
        elif kind in ("minres", "newton"):
            # A MINRES iteration: one J and CHEB - 1 products with P, and the
            # recurrences' vectors once (about twelve).
            it = case["iters"] * case.get("steps", 1)
            nbytes += it * (CHEB * apply_b + 12.0 * entry * n)
            flops += it * (CHEB * apply_f + 60.0 * n)
        elif kind == "continuation":
            it = 60.0 * 3 * (case["steps"] + 1)
            nbytes += it * (CHEB * apply_b + 12.0 * entry * n)
            flops += it * (CHEB * apply_f + 60.0 * n)
        elif kind == "eigen":
            it = 60.0 * (case["nev"] + 2)
            nbytes += it * (CHEB + 1) * apply_b
            flops += it * (CHEB + 1) * apply_f
        else:  # batch: the edges once for all lanes, FP32 inner vectors
            ln, it = case["lanes"], case["iters"] * case["steps"]
            nbytes += it * (5 * (16.0 * e + 28.0 * n * ln) + 96.0 * n * ln)
            flops += it * ln * (5 * apply_f + 60.0 * n)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------- the same in plain 64-bit torch
def _dot3(a, b):
    return (a * b).sum(-1)


def _unit_sign(s, area):
    return torch.where(torch.signbit(s), -area, area)


def _centre(p, q, r):
    """Circumcentre of triangles in space."""
    a, b, c = p - q, q - r, r - p
    w = 2.0 * _dot3(torch.linalg.cross(a, b), torch.linalg.cross(a, b))
    al = -_dot3(b, b) * _dot3(a, c) / w
    be = -_dot3(c, c) * _dot3(b, a) / w
    ga = -_dot3(a, a) * _dot3(c, b) / w
    return al[:, None] * p + be[:, None] * q + ga[:, None] * r


def _cell_weights(x):
    """Per cell and local edge the coefficient -|T| grad l_i . grad l_j (the
    one solution of the moment equations sum c e e^T = |T| I), and per cell
    and vertex its share of the circumcentric control volume."""
    if x.shape[1] == 3:
        pairs = [(0, 1), (1, 2), (2, 0)]
        area2 = torch.linalg.norm(torch.linalg.cross(x[:, 1] - x[:, 0], x[:, 2] - x[:, 0]), dim=1)
        c = [0.5 * _dot3(x[:, i] - x[:, 3 - i - j], x[:, j] - x[:, 3 - i - j]) / area2
             for i, j in pairs]
    else:
        pairs = [(0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3)]
        e = [x[:, k] - x[:, 0] for k in (1, 2, 3)]
        det = _dot3(e[0], torch.linalg.cross(e[1], e[2]))
        gr = [torch.linalg.cross(e[1], e[2]), torch.linalg.cross(e[2], e[0]),
              torch.linalg.cross(e[0], e[1])]
        gr = [v / det[:, None] for v in gr]
        gr = [-(gr[0] + gr[1] + gr[2])] + gr
        c = [-det.abs() / 6.0 * _dot3(gr[i], gr[j]) for i, j in pairs]
    share = [torch.zeros_like(c[0]) for _ in range(x.shape[1])]
    if x.shape[1] == 3:
        cc = _centre(x[:, 0], x[:, 1], x[:, 2])
        for i, j in pairs:
            mid, o = 0.5 * (x[:, i] + x[:, j]), x[:, 3 - i - j]
            side = _dot3(torch.linalg.cross(cc - x[:, i], mid - x[:, i]),
                         torch.linalg.cross(o - x[:, i], mid - x[:, i]))
            part = 0.25 * torch.linalg.norm(x[:, j] - x[:, i], dim=1) * _unit_sign(
                side, torch.linalg.norm(mid - cc, dim=1))
            share[i] = share[i] + part
            share[j] = share[j] + part
    else:
        sq = [_dot3(v, v)[:, None] for v in e]
        cc = x[:, 0] + (sq[0] * torch.linalg.cross(e[1], e[2]) + sq[1] * torch.linalg.cross(
            e[2], e[0]) + sq[2] * torch.linalg.cross(e[0], e[1])) / (2.0 * det[:, None])
        for i, j in pairs:
            o0, o1 = (x[:, k] for k in range(4) if k not in (i, j))
            mid = 0.5 * (x[:, i] + x[:, j])
            f0, f1 = _centre(x[:, i], x[:, j], o0), _centre(x[:, i], x[:, j], o1)
            gauge = torch.linalg.cross(o0 - mid, o1 - mid)
            norm = functools.partial(torch.linalg.norm, dim=1)
            cov = _unit_sign(_dot3(torch.linalg.cross(f0 - mid, cc - mid), gauge),
                             0.5 * norm(mid - f0) * norm(f0 - cc))
            cov = cov + _unit_sign(_dot3(torch.linalg.cross(cc - mid, f1 - mid), gauge),
                                   0.5 * norm(mid - f1) * norm(f1 - cc))
            part = norm(x[:, j] - x[:, i]) * cov / 6.0
            share[i] = share[i] + part
            share[j] = share[j] + part
    return pairs, c, share


class _Graph:
    """Edges, weights and control volumes of a mesh, and products with K."""

    def __init__(self, xyz, cells, ordered=False):
        self.n = n = len(xyz)
        x = torch.from_numpy(xyz).to(DEV)
        t = torch.from_numpy(cells.astype(np.int64)).to(DEV)
        pairs, c, share = _cell_weights(x[t])
        ends = torch.stack([torch.stack([t[:, i], t[:, j]], 1) for i, j in pairs], 1)
        key = (ends.amin(2) * n + ends.amax(2)).reshape(-1)
        c = torch.stack(c, 1).reshape(-1)
        uniq, inv = torch.unique(key, return_inverse=True)
        if ordered:  # edges in order of first appearance
            first = torch.full((len(uniq),), len(key), device=DEV).scatter_reduce(
                0, inv, torch.arange(len(key), device=DEV), "amin")
            order = torch.argsort(first)
            rank = torch.empty_like(order)
            rank[order] = torch.arange(len(order), device=DEV)
            uniq, inv = uniq[order], rank[inv]
        self.lo, self.hi = uniq // n, uniq % n
        self.alpha = torch.zeros(len(uniq), dtype=torch.float64, device=DEV).index_add_(0, inv, c)
        self.cv = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(
            0, t.reshape(-1), torch.stack(share, 1).reshape(-1))
        self.length = torch.linalg.norm(x[self.lo] - x[self.hi], dim=1)
        self.x = x

    def table(self):
        """Every vertex's neighbours, padded to the longest list."""
        A = torch.from_numpy(_potential(self.x.cpu().numpy())).to(DEV)
        at = _dot3(0.5 * (A[self.lo] + A[self.hi]), self.x[self.lo] - self.x[self.hi])
        row = torch.cat([self.lo, self.hi])
        row, by = torch.sort(row, stable=True)
        start = torch.searchsorted(row, torch.arange(self.n, device=DEV))
        place = torch.arange(len(row), device=DEV) - start[row]
        width = int(place.max()) + 1
        self.col = torch.zeros(self.n, width, dtype=torch.int64, device=DEV)
        self.w = torch.zeros(self.n, width, dtype=torch.float64, device=DEV)
        self.at = torch.zeros_like(self.w)
        self.col[row, place] = torch.cat([self.hi, self.lo])[by]
        self.w[row, place] = torch.cat([self.alpha, self.alpha])[by]
        self.at[row, place] = torch.cat([at, -at])[by]
        return self

    def set_mu(self, mu):
        self.k = torch.polar(self.w, -mu * self.at).neg_()
        self.diag, self.rowabs = self.w.sum(1), self.w.abs().sum(1)
        return self

    def K(self, x):
        return self.diag * x + (self.k * x[self.col]).sum(1)

    def F(self, x, g):
        return self.K(x) + self.cv * (g * x.abs() ** 2 - 1.0) * x

    def at_state(self, psi, g):
        """(V + 2 g |psi|^2, g psi^2, 2 g |psi|^2) weighted by the volumes."""
        r2 = psi.abs() ** 2
        return (self.cv * (2.0 * g * r2 - 1.0), g * self.cv * psi ** 2, 2.0 * g * self.cv * r2)

    def step(self, psi, b, g, iters, cheb):
        """iters preconditioned MINRES steps (Paige and Saunders) on J x = b."""
        vj, sq, vp = self.at_state(psi, g)
        a = self.diag + vp
        det = a ** 2 - sq.abs() ** 2
        hi = 1.0 + float((self.rowabs / (a - sq.abs())).max())
        theta, delta = 0.5 * (hi + hi / RATIO), 0.5 * (hi - hi / RATIO)

        def jac(x):
            return self.K(x) + vj * x + sq * x.conj()

        def dinv(r):
            return (a * r - sq * r.conj()) / det

        def prec(r):
            z = d = dinv(r) / theta
            rho = delta / theta
            for _ in range(1, cheb):
                new = 1.0 / (2.0 * theta / delta - rho)
                res = r - (self.K(z) + vp * z + sq * z.conj())
                d = new * rho * d + 2.0 * new / delta * dinv(res)
                z, rho = z + d, new
            return z

        def dot(p, q):
            return float((p.conj() * q).real.sum())

        x = torch.zeros_like(b)
        r1 = r2 = b
        y = prec(b)
        beta = math.sqrt(dot(b, y))
        oldb = dbar = eps = 0.0
        phibar, cs, sn = beta, -1.0, 0.0
        w = w2 = torch.zeros_like(b)
        for it in range(iters):
            v = y / beta
            u = jac(v)
            if it:
                u = u - (beta / oldb) * r1
            alfa = dot(v, u)
            u = u - (alfa / beta) * r2
            r1, r2 = r2, u
            y = prec(r2)
            oldb, beta = beta, math.sqrt(max(0.0, dot(r2, y)))
            olde = eps
            dl = cs * dbar + sn * alfa
            gbar = sn * dbar - cs * alfa
            eps, dbar = sn * beta, -cs * beta
            gamma = math.hypot(gbar, beta)
            cs, sn = gbar / gamma, beta / gamma
            phi, phibar = cs * phibar, sn * phibar
            w1, w2 = w2, w
            w = (v - olde * w1 - dl * w2) / gamma
            x = x + phi * w
        return x

    def dense(self, psi, g):
        """J(psi) as a real 2n x 2n matrix over (re, im)."""
        n = self.n
        K = torch.zeros(n, n, dtype=torch.complex128, device=DEV)
        rows = torch.arange(n, device=DEV)[:, None].expand_as(self.col)
        K.index_put_((rows, self.col), self.k, accumulate=True)
        vj, sq, _ = self.at_state(psi, g)
        K += torch.diag((self.diag + vj).to(torch.complex128))
        J = torch.empty(2 * n, 2 * n, dtype=torch.float64, device=DEV)
        J[:n, :n] = K.real + torch.diag(sq.real)
        J[:n, n:] = -K.imag + torch.diag(sq.imag)
        J[n:, :n] = K.imag + torch.diag(sq.imag)
        J[n:, n:] = K.real - torch.diag(sq.real)
        return J

    def newton(self, psi, g):
        """Full Newton steps with dense solves, orthogonal to the phase i psi."""
        for _ in range(30):
            f = self.F(psi, g)
            if float(torch.linalg.vector_norm(f)) <= 1e-13:
                break
            ph = 1j * psi
            q = torch.cat([ph.real, ph.imag])
            q = q / torch.linalg.vector_norm(q)
            d = torch.linalg.solve(self.dense(psi, g) + torch.outer(q, q),
                                   -torch.cat([f.real, f.imag]))
            psi = psi + torch.complex(d[:self.n], d[self.n:])
        return psi

    def gibbs(self, psi):
        return float(-(self.cv * psi.abs() ** 4).sum() / self.cv.sum())


def _graph(box):
    return _Graph(*_box(*box, seed=2)).table()


def _complex(x):
    return torch.from_numpy(x.view(np.complex128).copy()).to(DEV)


def _real(z):
    return torch.view_as_real(z).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("train", "infer"):
        return _exact_network(case, seed)
    boxes = _boxes(case)
    if kind == "mesh":
        G = _Graph(*_box(*boxes[0], seed=seed), ordered=True)
        return None, G.length, G.alpha * G.length, G.cv
    mu, g = _parameters(case, seed)
    if kind == "batch":
        out, lanes = [], case["lanes"]
        for k, box in enumerate(boxes):
            G = _graph(box)
            for i in range(k * lanes, (k + 1) * lanes):
                G.set_mu(float(mu[i]))
                psi = _complex(_near(G.n, g[i], seed, i))
                for _ in range(case["steps"]):
                    psi = psi + G.step(psi, -G.F(psi, g[i]), g[i], case["iters"], 5)
                out.append(_real(psi))
        return torch.cat(out)
    G, mu, g = _graph(boxes[0]), float(mu[0]), float(g[0])
    if kind == "operators":
        G.set_mu(mu)
        psi, phi = _complex(_random(G.n, seed, 0)), _complex(_random(G.n, seed, 1))
        vj, sq, _ = G.at_state(psi, g)
        kphi = G.K(phi)
        return _real(G.F(psi, g)), _real(kphi), _real(kphi + vj * phi + sq * phi.conj())
    if kind == "minres":
        G.set_mu(mu)
        psi = _complex(_near(G.n, g, seed, 0))
        return _real(G.step(psi, G.F(psi, g), g, case["iters"], CHEB)).cpu().numpy()
    if kind == "newton":
        G.set_mu(mu)
        psi = _complex(_near(G.n, g, seed, 0))
        for _ in range(case["steps"]):
            psi = psi + G.step(psi, -G.F(psi, g), g, case["iters"], CHEB)
        return _real(psi)
    psi = torch.full((G.n,), 1.0 / math.sqrt(g), dtype=torch.complex128, device=DEV)
    if kind == "continuation":
        energy = []
        for k in range(case["steps"] + 1):
            psi = G.set_mu((0.1 + mu) * k / case["steps"]).newton(psi, g)
            energy.append(G.gibbs(psi))
        return _phase_fixed(psi.cpu().numpy()), energy
    psi = G.set_mu(0.1 + mu).newton(psi, g)
    ph = 1j * psi
    q = torch.cat([ph.real, ph.imag])
    q = q / torch.linalg.vector_norm(q)
    J = G.dense(psi, g)
    Jq = J @ q
    J = J - torch.outer(q, Jq) - torch.outer(Jq, q) + (float(q @ Jq) + 1e6) * torch.outer(q, q)
    return np.linalg.eigvalsh(J.cpu().numpy())[:case["nev"]]


def _exact_network(case, seed):
    w, b = ([t.double().to(DEV).requires_grad_(case["kind"] == "train") for t in ts]
            for ts in _network(case, seed))

    def net(x):
        for k in range(len(w) - 1):
            x = torch.nn.functional.gelu(x @ w[k].T + b[k], approximate="tanh")
        return x @ w[-1].T + b[-1]

    if case["kind"] == "infer":
        x, _ = _samples(case["rows"], seed, 0)
        return torch.cat([net(part.double()) for part in x.split(1 << 17)])
    ps = w + b
    m = [torch.zeros_like(p) for p in ps]
    v = [torch.zeros_like(p) for p in ps]
    for k in range(case["steps"]):
        x, y = _samples(case["rows"], seed, k)
        loss = ((net(x.double()) - y.double()) ** 2).mean()
        grads = torch.autograd.grad(loss, ps)
        with torch.no_grad():
            for i, (p, d) in enumerate(zip(ps, grads)):
                m[i] = 0.9 * m[i] + 0.1 * d
                v[i] = 0.999 * v[i] + 0.001 * d * d
                p -= 1e-4 * (m[i] / (1 - 0.9 ** (k + 1))) / (
                    (v[i] / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    flat = torch.cat([p.detach().reshape(-1) for p in ps])
    return flat.cpu().numpy()
