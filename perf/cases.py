"""The assembly calls that performance is measured on: sizes, inputs and reference values.

A case is one mesh (or one batch of meshes) and one kind of call on it.  `prepare` does what a
finite-element program does once per mesh: coordinates and connectivity, DOF map, CRS graph,
Dirichlet lists, coefficients, state and the containers; `run` is one evaluation into those
containers through the package's Python entry points, as a Newton iteration or a time step makes
it.  `exact` assembles the same system with plain torch operations in 64 bits: its own numbering
(first touch in element order), its own graph and its own quadrature.
"""
import math

import numpy as np
import torch

import tianxin_amd as txa

_TOPO = {"hex8": txa.HEX8, "tet4": txa.TET4, "hex27": txa.HEX27}
_PREC = {"fp64": txa.FP64, "fp32": txa.FP32, "split": txa.SPLIT_BF16}

# Newmark (beta 1/4, gamma 1/2) with a millisecond step and light Rayleigh damping: the served
# time integration; the scalar transient form uses a backward Euler step of a tenth.
DT = 1e-3
NEWMARK = dict(alpha=0.5 / (0.25 * DT), beta=1.0, gamma2=1.0 / (0.25 * DT * DT))
RAYLEIGH = (0.01, 0.001)
EULER = dict(alpha=10.0, beta=1.0)
NU, RHO = 0.3, 1.2
SOURCE = {"diffusion": (1.0, 0.0, 0.0), "elasticity": (0.0, 0.0, -9.81)}

_engine = None


def _eng():
    global _engine
    if _engine is None:
        _engine = txa.Engine(0)
    return _engine


def _case(mesh, topo, physics, n, cells, precision="fp64", transient=False, want="fw", order="lattice", call="assemble"):
    return dict(mesh=mesh, topo=topo, physics=physics, nx=n[0], ny=n[1], nz=n[2], cells=cells, precision=precision,
                transient=transient, want=want, order=order, call=call)


def listed():
    dif, ela = "diffusion", "elasticity"
    return [
        # the ModelEvaluator call (f and W) of a small steady problem, where launches and latency count
        dict(name="poisson_hex8_32_model", **_case("brick", "hex8", dif, (32, 32, 32), "cube", call="model")),
        # the benchmark's workload: FP32 integration of a large structured Poisson problem
        dict(name="poisson_hex8_256_fp32", **_case("brick", "hex8", dif, (256, 256, 256), "cube", "fp32")),
        # an implicit time step on a distorted, ragged brick
        dict(name="poisson_hex8_jittered_step", **_case("brick", "hex8", dif, (161, 131, 97), "jittered", transient=True)),
        # the residual alone, as a line search or a matrix-free Krylov method asks for it
        dict(name="poisson_tet4_residual", **_case("brick", "tet4", dif, (97, 90, 83), "jittered", want="f")),
        # the smallest and the largest mesh of the served Newmark steps
        dict(name="elastic_hex8_18_newmark", **_case("brick", "hex8", ela, (18, 18, 18), "cube", transient=True)),
        dict(name="elastic_hex8_115_newmark", **_case("brick", "hex8", ela, (115, 115, 115), "cube", transient=True)),
        # the same step on distorted cells
        dict(name="elastic_hex8_jittered_newmark", **_case("brick", "hex8", ela, (96, 81, 72), "jittered", transient=True)),
        # quadratic elements: the FP64 form at a middle size, the matrix-core form at the benchmark's size
        dict(name="elastic_hex27_33_fp64", **_case("brick", "hex27", ela, (33, 33, 33), "jittered")),
        dict(name="elastic_hex27_64_split", **_case("brick", "hex27", ela, (64, 64, 64), "jittered", "split")),
        # meshes that arrive as connectivity, elements in no particular order
        dict(name="upload_poisson_hex8", **_case("upload", "hex8", dif, (100, 100, 100), "jittered", order="shuffled")),
        dict(name="upload_elastic_hex8", **_case("upload", "hex8", ela, (64, 61, 67), "jittered", transient=True,
                                                 order="shuffled")),
        # many small meshes in one launch
        dict(name="batch_128_mixed_fp32", mesh="batch", count=128, lo=8, hi=64, precision="fp32"),
    ]


def draw(rng):
    def size(lo, hi):
        """Three cell counts around a log-uniform mean, each its own."""
        n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return tuple(max(lo, min(hi, int(round(n * rng.uniform(0.75, 1.3))))) for _ in range(3))

    kind = rng.choice(["poisson", "poisson", "elastic", "elastic", "q2", "q2split", "upload_poisson", "upload_elastic", "batch"])
    cells = rng.choice(["cube", "jittered", "jittered"])
    transient = rng.random() < 0.5
    want = "f" if rng.random() < 0.2 else "fw"
    call = "model" if rng.random() < 0.3 else "assemble"
    order = rng.choice(["lattice", "shuffled"])
    prec = rng.choice(["fp64", "fp64", "fp32"])
    if kind == "poisson":
        topo = rng.choice(["hex8", "hex8", "tet4"])
        return _case("brick", topo, "diffusion", size(8, 240 if topo == "hex8" else 110), cells, prec, transient, want, call=call)
    if kind == "elastic":
        return _case("brick", "hex8", "elasticity", size(8, 115), cells, "fp64", transient, want, call=call)
    if kind == "q2":
        return _case("brick", "hex27", "elasticity", size(2, 44), cells, "fp64", transient, want, call=call)
    if kind == "q2split":
        return _case("brick", "hex27", "elasticity", size(2, 60), cells, "split", transient, "fw", call=call)
    if kind == "upload_poisson":
        return _case("upload", "hex8", "diffusion", size(8, 128), cells, prec, transient, want, order)
    if kind == "upload_elastic":
        return _case("upload", "hex8", "elasticity", size(8, 80), cells, "fp64", transient, want, order)
    lo = rng.choice([8, 12, 16])
    return dict(mesh="batch", count=int(round(math.exp(rng.uniform(math.log(2), math.log(128))))), lo=lo,
                hi=rng.randint(lo + 4, 64), precision=rng.choice(["fp32", "fp64"]))


# ------------------------------------------------------------------------------- meshes and inputs

def _coords(c, rng):
    """Lattice of the unit cube; jittered: interior vertices moved by up to a tenth of a cell."""
    n = (c["nx"], c["ny"], c["nz"])
    X = np.empty((n[2] + 1, n[1] + 1, n[0] + 1, 3))
    X[..., 0] = (np.arange(n[0] + 1) / n[0])[None, None, :]
    X[..., 1] = (np.arange(n[1] + 1) / n[1])[None, :, None]
    X[..., 2] = (np.arange(n[2] + 1) / n[2])[:, None, None]
    if c["cells"] == "jittered":
        inner = X[1:-1, 1:-1, 1:-1]
        off = rng.random(inner.shape) * 2.0 - 1.0
        inner += off * (0.1 / np.array(n))
    return X.reshape(-1, 3)


def _cell_verts(nx, ny, nz):
    """First vertex of each cell and the strides, cells x fastest."""
    i, j, k = np.arange(nx), np.arange(ny), np.arange(nz)
    base = (i[None, None, :] + (nx + 1) * (j[None, :, None] + (ny + 1) * k[:, None, None])).reshape(-1)
    return base.astype(np.int64), 1, nx + 1, (nx + 1) * (ny + 1)


# vertices of a cell as lattice offsets, in the element's order
_HEX = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]


def _hex_conn(nx, ny, nz):
    base, sx, sy, sz = _cell_verts(nx, ny, nz)
    return base[:, None] + np.array([a * sx + b * sy + d * sz for a, b, d in _HEX], np.int64)


def _shuffle(c, ne, rng):
    return rng.permutation(ne) if c["order"] == "shuffled" else None


def _inputs(nelem, ndofs, c, seed):
    """Coefficients (lognormal), state and rates, on the device."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda n: torch.rand(n, generator=g, device="cuda", dtype=torch.float64)   # noqa: E731
    nrm = torch.randn(nelem, generator=g, device="cuda", dtype=torch.float64)
    ela = c["physics"] == "elasticity"
    out = {"coef": torch.exp((0.3 if ela else 0.5) * nrm), "x": rnd(ndofs) * 2 - 1}
    if c["transient"]:
        out["xdot"] = rnd(ndofs) * 2 - 1
        if ela:
            out["xddot"] = rnd(ndofs) * 2 - 1
    return out


def _call_args(c):
    ela = c["physics"] == "elasticity"
    kw = dict(physics=txa.ELASTICITY if ela else txa.DIFFUSION, precision=_PREC[c["precision"]], src=SOURCE[c["physics"]])
    if ela:
        kw.update(nu=NU)
    if c["transient"]:
        kw.update(transient=True, rho=RHO, **(NEWMARK if ela else EULER))
        if ela:
            kw.update(rayleigh=RAYLEIGH)
    return kw


class State:
    """What one case holds between calls; the library's objects go when it does."""

    def __init__(self):
        self.owned = []   # destroyed last made first

    def __del__(self):
        for o in reversed(self.owned):
            try:
                o.destroy()
            except Exception:
                pass


def prepare(case, seed):
    return _prepare_batch(case, seed) if case["mesh"] == "batch" else _prepare_single(case, seed)


def _prepare_single(c, seed):
    rng = np.random.default_rng(seed)
    s = State()
    X = _coords(c, rng)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    nf = 3 if c["physics"] == "elasticity" else 1
    if c["mesh"] == "brick":
        m = _eng().brick(_TOPO[c["topo"]], nx, ny, nz, X)
    else:
        conn = _hex_conn(nx, ny, nz)
        perm = _shuffle(c, conn.shape[0], rng)
        m = _eng().upload(_TOPO[c["topo"]], conn if perm is None else conn[perm], X)
    s.owned.append(m)
    m.build_dofmap(nf)
    m.build_graph()
    # Dirichlet rows: the face x = 0, held at a given value
    if c["mesh"] == "brick":
        px = 2 * nx + 1 if c["topo"] == "hex27" else nx + 1
        lids = m.point_lids()[::px].reshape(-1)
    else:
        _, el = m.dofmap()
        conn = _hex_conn(nx, ny, nz)
        conn = conn if perm is None else conn[perm]
        of = np.empty((X.shape[0], nf), np.int32)
        of[conn.reshape(-1)] = el.reshape(-1, nf)
        lids = of[X[:, 0] == 0.0].reshape(-1)
    bc = torch.as_tensor(np.ascontiguousarray(lids), device="cuda")
    g = torch.linspace(0.0, 0.5, bc.numel(), device="cuda", dtype=torch.float64)
    inp = _inputs(m.nelem, m.ndofs, c, seed)
    s.mesh = m
    s.out = {"f": torch.zeros(m.ndofs, device="cuda", dtype=torch.float64)}
    if c["want"] == "fw":
        s.out["vals"] = torch.zeros(m.nnz, device="cuda", dtype=torch.float64)
    kw = _call_args(c)
    if c["call"] == "model":
        seeds = {k: kw.pop(k) for k in ("alpha", "beta", "gamma2") if k in kw}
        transient = kw.pop("transient", False)
        s.model = txa.Model(m, coef=inp["coef"], transient_support=transient, bc_lids=bc, bc_vals=g, **kw)
        s.owned.append(s.model)
        s.call = dict(x=inp["x"], x_dot=inp.get("xdot"), x_dot_dot=inp.get("xddot"), f=s.out["f"], W=s.out.get("vals"), **seeds)
    else:
        s.model = None
        s.call = dict(f=s.out["f"], vals=s.out.get("vals"), bc_lids=bc, bc_vals=g, **inp, **kw)
    s.batch = None
    return s


def _batch_meshes(c, seed):
    """(topology, cells per axis) of each mesh: sizes log-uniform, half hex8, half tet4, the same
    for every seed; the inputs differ."""
    r = np.random.default_rng(c["count"] * 1000003 + c["lo"] * 1009 + c["hi"])
    n = np.exp(r.uniform(math.log(c["lo"]), math.log(c["hi"] + 1), c["count"])).astype(int)
    t = r.random(c["count"]) < 0.5
    return [("tet4" if t[i] else "hex8", max(c["lo"], min(c["hi"], int(n[i])))) for i in range(c["count"])]


def _batch_case(c, topo, n):
    return _case("brick", topo, "diffusion", (n, n, n), "cube", c["precision"])


def _room(n):
    """Each mesh's part of the shared containers starts on a 256-byte line."""
    return (n + 31) // 32 * 32


def _prepare_batch(c, seed):
    s = State()
    meshes, faces = [], []
    for topo, n in _batch_meshes(c, seed):
        m = _eng().brick(_TOPO[topo], n, n, n, _coords(_batch_case(c, topo, n), None))
        m.build_dofmap(1)
        m.build_graph()
        s.owned.append(m)
        meshes.append(m)
        faces.append(torch.as_tensor(np.ascontiguousarray(m.point_lids()[::n + 1].reshape(-1)), device="cuda"))
    s.out = {"f": torch.zeros(sum(_room(m.ndofs) for m in meshes), device="cuda", dtype=torch.float64),
             "vals": torch.zeros(sum(_room(m.nnz) for m in meshes), device="cuda", dtype=torch.float64)}
    per, f0, v0 = [], 0, 0
    for i, (m, (topo, n)) in enumerate(zip(meshes, _batch_meshes(c, seed))):
        cc = _batch_case(c, topo, n)
        per.append(dict(f=s.out["f"][f0:f0 + m.ndofs], vals=s.out["vals"][v0:v0 + m.nnz], bc_lids=faces[i],
                        **_inputs(m.nelem, m.ndofs, cc, seed + 7919 * i), **_call_args(cc)))
        f0, v0 = f0 + _room(m.ndofs), v0 + _room(m.nnz)
    s.batch = txa.Batch(_eng(), meshes, precision=_PREC[c["precision"]])
    s.owned.append(s.batch)
    s.packed = s.batch.pack(per)
    s.keep = per
    s.model = None
    return s


def run(state):
    if state.batch is not None:
        state.batch.assemble(state.packed)
    elif state.model is not None:
        state.model.eval(**state.call)
    else:
        state.mesh.assemble(**state.call)
    return state.out


# ------------------------------------------------------------------------------------------- work

def _counts(c):
    """(elements, DOFs, nonzeros, vertices) of one mesh."""
    n = (c["nx"], c["ny"], c["nz"])
    cells, verts = n[0] * n[1] * n[2], (n[0] + 1) * (n[1] + 1) * (n[2] + 1)
    nf = 3 if c["physics"] == "elasticity" else 1
    if c["topo"] == "hex27":
        return cells, nf * math.prod(2 * v + 1 for v in n), nf * nf * math.prod(8 * v + 1 for v in n), verts
    if c["topo"] == "hex8":
        return cells, nf * verts, nf * nf * math.prod(3 * v + 1 for v in n), verts
    # six tets per cell: the edges are the lattice's, one diagonal per cell face, one per cell
    a, b, d = n
    edges = a * (b + 1) * (d + 1) + (a + 1) * b * (d + 1) + (a + 1) * (b + 1) * d
    faces = a * b * (d + 1) + a * (b + 1) * d + (a + 1) * b * d
    return 6 * cells, nf * verts, nf * nf * (verts + 2 * (edges + faces + cells)), verts


def work(case):
    """Coordinates, coefficients and state read once, f and the matrix written once; connectivity
    where the mesh has no lattice.  The operations: the symmetric element matrix by quadrature, or the
    residual alone."""
    if case["mesh"] == "batch":
        parts = [work(_batch_case(case, t, n)) for t, n in _batch_meshes(case, 0)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    ne, nd, nnz, nv = _counts(case)
    ela = case["physics"] == "elasticity"
    states = 1 if not case["transient"] else (3 if ela else 2)
    b = 24 * nv + 8 * ne + 8 * nd * (states + 1)
    if case["mesh"] == "upload":
        b += 32 * ne
    nb, nq = {"hex8": (8, 8), "tet4": (4, 1), "hex27": (27, 27)}[case["topo"]]
    nf = 3 if ela else 1
    if case["want"] == "fw":
        b += 8 * nnz
        # hex8 diffusion: the sum-factorised form; the others the symmetric gradient products
        fl = {("hex8", False): 1300, ("tet4", False): 150}.get((case["topo"], ela), 3 * nb * (3 * nb + 1) * nq + 36 * nb * nb)
    else:
        fl = nq * (nb * 3 * (2 + 2 * nf) + 60)
    return {"bytes": float(b), "flops": float(fl * ne)}


# ------------------------------------------------------------------------------------------ exact

_TETS = [(0, 2, 3, 6), (0, 3, 7, 6), (0, 7, 4, 6), (0, 5, 6, 4), (1, 5, 6, 0), (1, 6, 2, 0)]   # hex vertex order
_Q2 = [(0, 0, 0), (2, 0, 0), (2, 2, 0), (0, 2, 0), (0, 0, 2), (2, 0, 2), (2, 2, 2), (0, 2, 2),
       (1, 0, 0), (2, 1, 0), (1, 2, 0), (0, 1, 0), (1, 0, 2), (2, 1, 2), (1, 2, 2), (0, 1, 2),
       (0, 0, 1), (2, 0, 1), (2, 2, 1), (0, 2, 1),
       (1, 0, 1), (2, 1, 1), (1, 2, 1), (0, 1, 1), (1, 1, 0), (1, 1, 2), (1, 1, 1)]


def _lagrange(order, xi):
    if order == 1:
        return [0.5 * (1 - xi), 0.5 * (1 + xi)], [-0.5, 0.5]
    return [0.5 * xi * (xi - 1), 1 - xi * xi, 0.5 * xi * (xi + 1)], [xi - 0.5, -2 * xi, xi + 0.5]


def _tables(topo):
    """(basis [nb, nq], its gradients [nb, nq, 3], geometry gradients [nv, nq, 3], weights [nq])."""
    if topo == "tet4":   # the degree-2 rule with four points
        a, b = (5 + 3 * math.sqrt(5)) / 20, (5 - math.sqrt(5)) / 20
        pts = [(b, b, b), (a, b, b), (b, a, b), (b, b, a)]
        N = np.array([[1 - sum(p) for p in pts]] + [[p[d] for p in pts] for d in range(3)])
        dN = np.zeros((4, 4, 3))
        dN[0] = -1.0
        for d in range(3):
            dN[d + 1, :, d] = 1.0
        return N, dN, dN, np.full(4, 1 / 24)
    order = 2 if topo == "hex27" else 1
    x, w = np.polynomial.legendre.leggauss(order + 1)
    nodes = _Q2 if order == 2 else _HEX
    pts = [(i, j, k) for k in range(order + 1) for j in range(order + 1) for i in range(order + 1)]

    def tab(nodes, order):
        L = [_lagrange(order, v) for v in x]
        N = np.array([[L[p[0]][0][a] * L[p[1]][0][b] * L[p[2]][0][d] for p in pts] for a, b, d in nodes])
        dN = np.array([[[L[p[0]][1][a] * L[p[1]][0][b] * L[p[2]][0][d], L[p[0]][0][a] * L[p[1]][1][b] * L[p[2]][0][d],
                         L[p[0]][0][a] * L[p[1]][0][b] * L[p[2]][1][d]] for p in pts] for a, b, d in nodes])
        return N, dN

    N, dN = tab(nodes, order)
    return N, dN, tab(_HEX, 1)[1], np.array([w[i] * w[j] * w[k] for i, j, k in pts])


def exact(case, seed):
    if case["mesh"] == "batch":
        fs, vs = [], []
        for i, (topo, n) in enumerate(_batch_meshes(case, seed)):
            r = _exact_single(_batch_case(case, topo, n), seed, seed + 7919 * i, held=0.0)
            for out, v in ((fs, r["f"]), (vs, r["vals"])):
                out.append(torch.zeros(_room(v.numel()), device=v.device, dtype=v.dtype))
                out[-1][:v.numel()] = v
        return {"f": torch.cat(fs), "vals": torch.cat(vs)}
    nb = {"hex8": 8, "tet4": 4, "hex27": 27}[case["topo"]]
    if _counts(case)[0] * nb * nb > 400_000_000:   # the largest: too long a sort
        return None
    return _exact_single(case, seed, seed)


def _exact_single(c, mesh_seed, input_seed, held=0.5):
    dev, f64 = "cuda", torch.float64
    rng = np.random.default_rng(mesh_seed)
    X = _coords(c, rng)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    geo = _hex_conn(nx, ny, nz)
    perm = _shuffle(c, geo.shape[0], rng)
    geo = geo if perm is None else geo[perm]
    if c["topo"] == "tet4":
        geo = geo[:, np.array(_TETS)].reshape(-1, 4)
    geo = torch.as_tensor(geo, device=dev)
    Xd = torch.as_tensor(X, device=dev)
    if c["topo"] == "hex27":
        q = [torch.arange(n, device=dev) for n in (nx, ny, nz)]
        px, py = 2 * nx + 1, 2 * ny + 1
        base = (2 * q[0][None, None, :] + px * (2 * q[1][None, :, None] + py * 2 * q[2][:, None, None])).reshape(-1)
        node = base[:, None] + torch.tensor([a + px * (b + py * d) for a, b, d in _Q2], device=dev)
        npts = px * py * (2 * nz + 1)
        on_face = torch.arange(npts, device=dev) % px == 0
    else:
        node, npts = geo, X.shape[0]
        on_face = Xd[:, 0] == 0.0
    ne, nb = node.shape
    nf = 3 if c["physics"] == "elasticity" else 1
    # numbering: points in the order in which the elements' nodes first touch them
    flat = node.reshape(-1)
    first = torch.full((npts,), flat.numel(), device=dev, dtype=torch.int64)
    first.scatter_reduce_(0, flat, torch.arange(flat.numel(), device=dev), "amin")
    lid = torch.empty(npts, device=dev, dtype=torch.int64)
    lid[torch.argsort(first)] = torch.arange(npts, device=dev)
    el = lid[node]
    inp = _inputs(ne, nf * npts, c, input_seed)
    u, v, a = (inp.get(k) for k in ("x", "xdot", "xddot"))
    N, dN, gd, w = (torch.as_tensor(t, device=dev) for t in _tables(c["topo"]))
    f = torch.zeros(nf * npts, device=dev, dtype=f64)
    vals = None
    if c["want"] == "fw":
        keys = []
        step = max(1, 60_000_000 // (nb * nb))
        for e0 in range(0, ne, step):
            p = el[e0:e0 + step]
            keys.append(torch.unique((p[:, :, None] * npts + p[:, None, :]).reshape(-1)))
        keys = torch.unique(torch.cat(keys))
        row = torch.searchsorted(keys, torch.arange(npts + 1, device=dev) * npts)   # row starts of the point graph
        vals = torch.zeros(nf * nf * keys.numel(), device=dev, dtype=f64)
    src = torch.tensor(SOURCE[c["physics"]][:nf], device=dev, dtype=f64)
    rho = RHO if c["transient"] else 1.0
    seeds = (NEWMARK if nf == 3 else EULER) if c["transient"] else {}
    al, be, g2 = seeds.get("alpha", 0.0), seeds.get("beta", 1.0), seeds.get("gamma2", 0.0)
    chunk = max(1, 24_000_000 // (nf * nb) ** 2)
    dof = torch.arange(nf, device=dev)
    for e0 in range(0, ne, chunk):
        p, k = el[e0:e0 + chunk], inp["coef"][e0:e0 + chunk]
        J = torch.einsum("evd,vqm->eqdm", Xd[geo[e0:e0 + chunk]], gd)
        cof = torch.linalg.cross(J[..., [1, 2, 0]], J[..., [2, 0, 1]], dim=2)   # det J times J^-T
        det = (J[..., 0] * cof[..., 0]).sum(-1)
        wm = w * det * torch.sign(det[:, :1])
        G = torch.einsum("eqdm,aqm->eqad", cof / det[..., None, None], dN)
        M = rho * torch.einsum("eq,aq,bq->eab", wm, N, N)
        F = torch.einsum("eq,aq,i->eai", wm, N, src)
        E = G.shape[0]
        A = (G * wm[:, :, None, None]).reshape(E, G.shape[1], -1)
        T = torch.bmm(A.transpose(1, 2).contiguous(), G.reshape(E, G.shape[1], -1)).reshape(E, nb, 3, nb, 3)
        tr = T.diagonal(dim1=2, dim2=4).sum(-1)
        eye = torch.eye(nf, device=dev, dtype=f64)
        Mf = M[:, :, None, :, None] * eye[:, None, :]
        if nf == 1:
            K = (k[:, None, None] * tr)[:, :, None, :, None]
            C = Mf
        else:
            lam, mu = k * NU / ((1 + NU) * (1 - 2 * NU)), k / (2 * (1 + NU))
            q = (slice(None), None, None, None, None)
            K = lam[q] * T + mu[q] * (T.permute(0, 1, 4, 3, 2) + tr[:, :, None, :, None] * eye[:, None, :])
            C = RAYLEIGH[0] * Mf + RAYLEIGH[1] * K
        d = nf * p[:, :, None] + dof
        R = torch.einsum("eaibj,ebj->eai", K, u[d]) - F
        Je = be * K
        if c["transient"]:
            R = R + torch.einsum("eaibj,ebj->eai", C, v[d])
            Je = Je + al * C
            if nf == 3:
                R = R + torch.einsum("eaibj,ebj->eai", Mf, a[d])
                Je = Je + g2 * Mf
        f.index_add_(0, d.reshape(-1), R.reshape(-1))
        if vals is not None:
            pos = torch.searchsorted(keys, (p[:, :, None] * npts + p[:, None, :]).reshape(-1)).reshape(E, nb, nb)
            r0 = row[p][:, :, None]
            deg = (row[p + 1] - row[p])[:, :, None]
            at = (nf * nf * r0 + nf * (pos - r0))[:, :, None, :, None] + (nf * deg)[:, :, None, :, None] * dof[:, None, None] + dof
            vals.index_add_(0, at.reshape(-1), Je.expand(E, nb, nf, nb, nf).reshape(-1))
    # Dirichlet rows, listed in the order of the lattice points of the face (uploads: of the vertices)
    rows = (nf * lid[on_face][:, None] + dof).reshape(-1)
    g = torch.linspace(0.0, held, rows.numel(), device=dev, dtype=f64) if held else torch.zeros(rows.numel(), device=dev, dtype=f64)
    f[rows] = u[rows] - g
    out = {"f": f}
    if vals is not None:
        pt, fi = rows // nf, rows % nf
        r0, deg = row[pt], row[pt + 1] - row[pt]
        start, n = nf * nf * r0 + fi * nf * deg, nf * deg
        of = torch.repeat_interleave(torch.arange(rows.numel(), device=dev), n)
        off = torch.arange(of.numel(), device=dev) - (torch.cumsum(n, 0) - n)[of]
        vals[start[of] + off] = 0.0
        diag = torch.searchsorted(keys, pt * npts + pt)
        vals[start + nf * (diag - r0) + fi] = 1.0
        out["vals"] = vals
    return out
