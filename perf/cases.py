"""The work that programs ask of this framework, as cases that can be timed and checked.

A case is a dict of plain values.  `listed` gives the cases by name, `draw` more of the same
ranges, `prepare` what a program holds before the call (its operator, solver, coefficient
fields), `run` one pass through the public API, `work` the bytes and operations that pass cannot
do without, and `exact` the same results from plain torch in 64 bits (its own numbering, element
matrices and conjugate gradients; nothing of fempar_amd).

Kinds of case
  poisson     assemble -div(k grad u) = f on a box mesh and solve it by Jacobi-PCG, u to the host
  new_mesh    the same, from the mesh on: triangulation, numbering, pattern, assembly, solve
  mapped      Poisson on a mesh whose vertices were moved (every cell its own map)
  elasticity  vector Q1 linear elasticity, clamped on x = x_min
  multifield  two coupled fields, Q2 and Q1, in two blocks
  batch       many small independent Poisson problems in one launch
  serve       a burst of elasticity requests through the request server
"""
import itertools
import math

import numpy as np
import torch

import fempar_amd as F

RTOL = 1e-10
_env = None


def environment():
    global _env
    if _env is None:
        _env = F.environment_t(0)   # one per program: device and stream
    return _env


# ------------------------------------------------------------------------ cases ---

def _poisson(name, n, order=1, precision="FP64", k="sin3", bc="boundary", kind="poisson"):
    n = list(n) + [1] * (3 - len(n)) if len(n) == 2 else list(n)
    dim = 2 if n[2] == 1 else 3
    return {"name": name, "kind": kind, "dim": dim, "nx": n[0], "ny": n[1], "nz": n[2], "order": order,
            "precision": precision, "k": k, "bc": bc}


def listed():
    return [
        # the tutorial and test size of the drivers (test_poisson): a few hundred unknowns, launches and latency
        _poisson("poisson2d_q1_32", (32, 32)),
        # a large planar problem, odd sizes, coefficient and source evaluated by the caller at the quadrature points
        _poisson("poisson2d_q1_1001x700_qpoint", (1001, 700), k="qpoint"),
        # the headline benchmark: assembly + CG at 128^3 Q1 in the drop-in precision
        _poisson("poisson3d_q1_128", (128, 128, 128)),
        # and in the FP32-refined precision
        _poisson("poisson3d_q1_128_refined", (128, 128, 128), precision="FP32_REFINED"),
        # a first solve on a mesh just made (mesh adaptation, parameter studies of the geometry): set-up counts;
        # ragged sizes, Dirichlet on one face only, a cell-wise random coefficient
        _poisson("poisson3d_q1_new_mesh_77x53x61", (77, 53, 61), k="cell", bc="x0", kind="new_mesh"),
        # second order elements, 64^3 cells, as the benchmark's Q2 configuration
        _poisson("poisson3d_q2_64", (64, 64, 64), order=2),
        # the largest scalar problem of the benchmark: 192^3, log-normal coefficient of high contrast, refined
        _poisson("poisson3d_q1_192_field_refined", (192, 192, 192), precision="FP32_REFINED", k="cell"),
        # graded and deformed meshes: general cells, odd sizes
        _poisson("mapped3d_q1_57x49x65", (57, 49, 65), k="const", kind="mapped"),
        # structural analysis: vector Q1, one clamped face
        {"name": "elasticity3d_40x33x47_refined", "kind": "elasticity", "nx": 40, "ny": 33, "nz": 47,
         "precision": "FP32_REFINED"},
        # velocity-pressure shaped pair of fields, block CG
        {"name": "multifield_q2q1_32", "kind": "multifield", "n": 32},
        # a batch of uneven small problems, 70 % planar 16..256, 30 % solid 8..48, as the batched benchmark's mix
        {"name": "batch_512", "kind": "batch", "count": 512, "mix": 4096},
        # a burst of ten elasticity requests of mixed sizes, as the serving benchmark draws them
        {"name": "serve_10", "kind": "serve", "count": 10, "lo": 8, "hi": 56, "mix": 5000},
    ]


def _spread(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["q1_3d", "q1_3d", "q1_3d", "q1_2d", "q2", "q2", "new_mesh", "mapped", "elasticity",
                       "multifield", "batch", "serve"])
    precision = rng.choice(["FP64", "FP32_REFINED"])
    bc = rng.choice(["boundary", "boundary", "x0"])

    def box(lo, hi):   # sides near one size, seldom equal
        s = _spread(rng, lo, hi)
        return tuple(max(2, min(hi, int(s * rng.uniform(0.75, 1.25)))) for _ in range(3))

    if kind == "q1_3d":
        c = _poisson("", box(10, 150), precision=precision, k=rng.choice(["sin3", "cell", "const"]), bc=bc)
    elif kind == "q1_2d":
        s = _spread(rng, 16, 1200)
        c = _poisson("", (s, max(8, int(s * rng.uniform(0.5, 1.0)))), precision=precision,
                     order=rng.choice([1, 1, 2]) if s < 500 else 1, k=rng.choice(["sin3", "cell", "qpoint"]), bc=bc)
    elif kind == "q2":
        c = _poisson("", box(5, 52), order=2, precision=precision, k=rng.choice(["sin3", "cell", "const"]), bc=bc)
    elif kind == "new_mesh":
        order = rng.choice([1, 2])
        c = _poisson("", box(6, 80 if order == 1 else 36), order=order, precision=precision,
                     k=rng.choice(["sin3", "cell", "const"]), bc=bc, kind="new_mesh")
    elif kind == "mapped":
        c = _poisson("", box(8, 80), precision=precision, k="const", kind="mapped")
    elif kind == "elasticity":
        b = box(6, 52)
        c = {"kind": "elasticity", "nx": b[0], "ny": b[1], "nz": b[2], "precision": precision}
    elif kind == "multifield":
        c = {"kind": "multifield", "n": _spread(rng, 5, 36)}
    elif kind == "batch":
        c = {"kind": "batch", "count": _spread(rng, 8, 500), "mix": rng.randrange(1 << 20)}
    else:
        c = {"kind": "serve", "count": _spread(rng, 1, 10), "lo": 8, "hi": 48, "mix": rng.randrange(1 << 20)}
    c.pop("name", None)
    return c


# ----------------------------------------------------------------------- inputs ---

def _cells(case):
    return (case["nx"], case["ny"], case["nz"])[: case.get("dim", 3)]


def _gen(seed, salt=0):
    return np.random.default_rng([int(seed), salt])


def _field(n, seed, sigma=1.5, ell=0.1):
    """k per cell = exp of a Gaussian random field (squared-exponential correlation of length ell,
    standard deviation sigma), x fastest: a log-normal permeability."""
    dev = "cuda"
    m = [v + 1 for v in reversed(n)]
    g = torch.Generator(device=dev).manual_seed(int(seed) % (1 << 31))
    w = torch.randn(m, generator=g, device=dev, dtype=torch.float64)
    k2 = torch.zeros([1] * len(m), device=dev, dtype=torch.float64)
    for a, s in enumerate(m):
        f = 2 * math.pi * torch.fft.fftfreq(s, d=1.0 / (s - 1), device=dev, dtype=torch.float64)
        k2 = k2 + (f ** 2).reshape([-1 if b == a else 1 for b in range(len(m))])
    z = torch.fft.ifftn(torch.fft.fftn(w) * torch.exp(-(ell ** 2) * k2 / 4.0)).real
    z = (z - z.mean()) / z.std() * sigma
    for a in range(len(m)):   # mean over the cell's vertices
        z = 0.5 * (z.narrow(a, 0, m[a] - 1) + z.narrow(a, 1, m[a] - 1))
    return torch.exp(z).reshape(-1).cpu().numpy()


def _waves(seed, salt):
    r = _gen(seed, salt)
    return r.uniform(-0.5, 0.5, 4), r.integers(1, 5, (4, 3)), r.uniform(0, 2 * math.pi, (4, 3))


def _wave(x, modes):
    amp, freq, phase = modes
    s = 0.0
    for a, f, p in zip(amp, freq, phase):
        t = a
        for d in range(x.shape[-1]):
            t = t * np.sin(math.pi * f[d] * x[..., d] + p[d])
        s = s + t
    return s


def _moved_vertices(n, seed):
    """Uniform vertices of the unit box moved by a smooth map and a jitter of a tenth of a cell."""
    r = _gen(seed, 7)
    grids = np.meshgrid(*[np.arange(k + 1) / k for k in n], indexing="ij")
    x = np.stack([g.transpose().ravel() for g in grids], axis=1)
    modes = [_waves(seed, 20 + d) for d in range(len(n))]
    bump = np.prod(np.sin(math.pi * x), axis=1)
    moved = np.stack([x[:, d] + 0.05 * bump * _wave(x, modes[d]) for d in range(len(n))], axis=1)
    inner = np.all((x > 1e-9) & (x < 1 - 1e-9), axis=1)[:, None]
    return moved + inner * r.uniform(-0.1, 0.1, x.shape) / np.array(n)


def _data(case, seed):
    """Coefficient and source of a Poisson case, from the seed."""
    d = {"f0": float(_gen(seed, 1).uniform(0.5, 2.0)), "k0": float(_gen(seed, 2).uniform(0.5, 2.0))}
    if case["k"] == "cell":
        d["k_cell"] = _field(_cells(case), seed)
    elif case["k"] == "qpoint":
        km, fm = _waves(seed, 3), _waves(seed, 4)
        d["k_fn"] = lambda x: np.exp(_wave(x, km))
        d["f_fn"] = lambda x: d["f0"] + _wave(x, fm)
    if case["kind"] == "mapped":
        d["vertices"] = _moved_vertices(_cells(case), seed)
    return d


def _batch_problems(case, seed):
    """70 % planar n x n with n log-uniform in [16, 256], 30 % solid n^3 with n log-uniform in [8, 48]; the
    sizes belong to the case, coefficients and sources to the seed."""
    s, v = _gen(case["mix"], 5), _gen(seed, 6)
    out = []
    for _ in range(case["count"]):
        planar = s.random() < 0.7
        lo, hi = (16, 256) if planar else (8, 48)
        n = int(round(math.exp(s.uniform(math.log(lo), math.log(hi)))))
        out.append((2 if planar else 3, n, float(v.uniform(0.1, 10.0)), float(v.uniform(0.5, 2.0))))
    return out


def _serve_requests(case, seed):
    s, v = _gen(case["mix"], 8), _gen(seed, 9)
    return [(int(round(math.exp(s.uniform(math.log(case["lo"]), math.log(case["hi"]))))),
             float(v.uniform(1.0, 200.0)), float(v.uniform(0.2, 0.45))) for _ in range(case["count"])]


def _elastic(seed):
    r = _gen(seed, 10)
    return float(r.uniform(1.0, 200.0)), float(r.uniform(0.2, 0.45)), tuple(float(t) for t in r.uniform(-1.0, 1.0, 3))


def _two_fields(seed):
    r = _gen(seed, 11)
    return [float(t) for t in r.uniform(0.5, 2.0, 2)], float(r.uniform(0.2, 2.0)), [float(t) for t in r.uniform(0.5, 2.0, 2)]


# ---------------------------------------------------------------- through the API ---

def _solver(op, precision="FP64"):
    s = F.iterative_linear_solver_t().create(environment())
    s.set_type_from_string("CG")
    s.set_parameters_from_pl({"ILS_RTOL": RTOL, "ILS_MAX_NUM_ITERATIONS": 20000, "FEMHIP_PRECISION": precision})
    s.set_operators(op.get_tangent(), F.jacobi_preconditioner_t(op))
    return s


def _triangulation(n, vertices=None):
    return F.serial_triangulation_t().create(environment(), {
        "STRUCT_HEX_MESH_GENERATOR_NUM_DIMS": len(n), "STRUCT_HEX_MESH_GENERATOR_NUM_CELLS_X_DIM": list(n),
        "STRUCT_HEX_MESH_GENERATOR_DOMAIN_LIMITS": [0, 1, 0, 1, 0, 1]}, vertex_coordinates=vertices)


def _poisson_operator(case, d):
    fes = F.serial_fe_space_t().create(_triangulation(_cells(case), d.get("vertices")), order=case["order"],
                                       dirichlet=case["bc"])
    if case["k"] == "qpoint":
        di = F.poisson_discrete_integration_t(k=d["k_fn"], f=d["f_fn"])
    else:
        di = F.poisson_discrete_integration_t(k=case["k"], k0=d["k0"], k_cell=d.get("k_cell"), f="const", f0=d["f0"])
    op = F.fe_affine_operator_t()
    op.create("CSR", [True], fes, di)
    return op


def prepare(case, seed):
    kind = case["kind"]
    if kind == "new_mesh":
        return {"kind": kind, "case": case, "data": _data(case, seed)}
    if kind in ("poisson", "mapped"):
        op = _poisson_operator(case, _data(case, seed))
        return {"kind": kind, "op": op, "solver": _solver(op, case["precision"])}
    if kind == "elasticity":
        E, nu, body = _elastic(seed)
        fes = F.serial_fe_space_t().create(_triangulation(_cells(case)), order=1, num_components=3, dirichlet="x0")
        op = F.fe_affine_operator_t()
        op.create("CSR", [True], fes, F.linear_elasticity_discrete_integration_t(E, nu, body))
        return {"kind": kind, "op": op, "solver": _solver(op, case["precision"])}
    if kind == "multifield":
        kappa, sigma, f = _two_fields(seed)
        tria = _triangulation([case["n"]] * 3)
        spaces = [F.serial_fe_space_t().create(tria, order=2), F.serial_fe_space_t().create(tria, order=1)]
        op = F.block_fe_affine_operator_t()
        op.create("CSR", [False], spaces, F.block_layout_t().create(2, [1, 2]),
                  F.coupled_diffusion_discrete_integration_t(kappa, sigma, f))
        return {"kind": kind, "op": op, "solver": _solver(op)}
    if kind == "batch":
        problems = _batch_problems(case, seed)
        return {"kind": kind, "count": len(problems), "batch": F.batch_t(environment(), problems, rtol=RTOL)}
    requests = _serve_requests(case, seed)
    return {"kind": kind, "requests": requests,
            "server": F.serve_t(environment(), hbm_budget_bytes=16 << 30, max_active=8, setup_threads=8, rtol=RTOL)}


def run(state):
    kind = state["kind"]
    if kind == "new_mesh":
        case = state["case"]
        op = _poisson_operator(case, state["data"])
        op.compute()
        solver = _solver(op, case["precision"])
        solver.solve_resident()
        return solver.get_solution()
    if kind == "batch":
        b = state["batch"]
        b.assemble()
        b.solve()
        return np.concatenate([b.get_solution(i) for i in range(state["count"])])
    if kind == "serve":
        srv = state["server"]
        tickets = [srv.submit(n, E, nu) for n, E, nu in state["requests"]]
        out = []
        for t in tickets:
            srv.wait(t)
            out.append(srv.get_solution(t))
            srv.release(t)
        return out
    op, solver = state["op"], state["solver"]
    op.compute()
    if kind == "multifield":
        return solver.solve()
    solver.solve_resident()
    return solver.get_solution()


# ------------------------------------------------------------------------- work ---

def _sizes(case):
    """(unknowns, cells, iterations, stored matrix entries, bytes a coefficient) of a single-operator case."""
    n = _cells(case)
    p, dim = case.get("order", 1), len(n)
    cells = math.prod(n)
    if case["kind"] == "elasticity":
        nodes = n[0] * (n[1] + 1) * (n[2] + 1)
        return 3 * nodes, cells, 25.0 * max(n), 81 * 3 * nodes, 0
    inner = [p * v - 1 for v in n] if case["bc"] == "boundary" else [p * n[0]] + [p * v + 1 for v in n[1:]]
    rows = math.prod(inner)
    per = (3 if p == 1 else 4) ** dim   # entries of a row: 9 / 27 for Q1, about 16 / 64 on average for Q2
    its = (1.9 if p == 1 else 4.8) * max(n) * (2.4 if case["k"] == "cell" else 1.0) * (1.8 if case["bc"] == "x0" else 1.0)
    return rows, cells, its, per * rows, {"cell": 8.0, "qpoint": 8.0 * 2 * 2 ** dim}.get(case["k"], 0.0)


def work(case):
    """A CG iteration cannot do without reading and writing x, r and p once (6 words a row; 32-bit words in the
    refined precision) and reading the cells' coefficients; the assembly writes the matrix and the right-hand
    side once, and the solution goes to the host once."""
    kind = case["kind"]
    if kind == "batch":
        by = fl = 0.0
        for dim, n, _, _ in _batch_problems(case, 0):
            rows = (n - 1) ** dim
            by += rows * (24.0 * 1.5 * n + 8.0 * 3 ** dim + 16.0)
            fl += rows * 2.0 * 3 ** dim * 1.5 * n
        return {"bytes": by, "flops": fl}
    if kind == "serve":
        by = fl = 0.0
        for n, _, _ in _serve_requests(case, 0):
            rows = 3 * n * (n + 1) ** 2
            by += rows * (24.0 * 6 * n + 16.0)
            fl += rows * 2.0 * 81 * 6 * n
        return {"bytes": by, "flops": fl}
    if kind == "multifield":
        n = case["n"]
        rows = (2 * n - 1) ** 3 + (n - 1) ** 3
        nnz = 92.0 * rows
        its = 4.2 * n
        return {"bytes": its * 48.0 * rows + 8.0 * nnz + 16.0 * rows, "flops": its * 2.0 * nnz}
    rows, cells, its, nnz, coef = _sizes(case)
    word = 8.0 if case["precision"] == "FP64" else 4.0
    by = its * (6 * word * rows + coef * cells) + 8.0 * nnz + 16.0 * rows + coef * cells
    if kind == "mapped":
        by += 24.0 * cells
    return {"bytes": by, "flops": its * 2.0 * nnz + 10.0 * nnz}


# ------------------------------------------------------- the same in plain 64 bits ---

DEV = "cuda"


def _gauss(m):
    x, w = np.polynomial.legendre.leggauss(m)
    return x, w


def _shape_tables(dim, order, m):
    """Lagrange shape values (nodes, points) and reference gradients (nodes, points, dim) on [-1, 1]^dim at the
    m^dim Gauss points, and the weights; node and point indices x fastest."""
    x, w = _gauss(m)
    t = np.linspace(-1, 1, order + 1)
    v = np.empty((order + 1, m))
    dv = np.empty((order + 1, m))
    for i in range(order + 1):
        poly = np.poly1d([1.0])
        for j in range(order + 1):
            if j != i:
                poly = poly * np.poly1d([1.0, -t[j]]) / (t[i] - t[j])
        v[i], dv[i] = poly(x), poly.deriv()(x)
    nodes = [tuple(reversed(a)) for a in itertools.product(range(order + 1), repeat=dim)]
    points = [tuple(reversed(a)) for a in itertools.product(range(m), repeat=dim)]
    S = np.array([[math.prod(v[a[d], q[d]] for d in range(dim)) for q in points] for a in nodes])
    G = np.array([[[math.prod((dv if e == d else v)[a[e], q[e]] for e in range(dim)) for d in range(dim)]
                   for q in points] for a in nodes])
    W = np.array([math.prod(w[i] for i in q) for q in points])
    xi = np.array([[x[i] for i in q] for q in points])
    return S, G, W, xi


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV, dtype=torch.float64)


def _numbering(n, order, ncomp, bc):
    """Row of every (cell, local DOF), -1 where fixed, and the number of rows: DOFs numbered as the cells (x
    fastest) first touch them, a cell's interior before its vertices, edges and faces, components outermost
    within an entity; local DOF = component * nodes + node."""
    dim, np1 = len(n), order + 1
    nodes = [tuple(reversed(a)) for a in itertools.product(range(np1), repeat=dim)]
    key = []
    for a in nodes:
        typ = sum(1 << d for d in range(dim) if 0 < a[d] < order)
        anc = sum(1 << d for d in range(dim) if a[d] == order)
        dims = bin(typ).count("1")
        key.append((-1, 0) if dims == dim else (dims, (typ << dim) | anc))
    seq = sorted(range(ncomp * len(nodes)), key=lambda l: (key[l % len(nodes)], l))
    rank = torch.empty(len(seq), dtype=torch.int64, device=DEV)
    rank[torch.tensor(seq, device=DEV)] = torch.arange(len(seq), device=DEV)
    fine = [order * v + 1 for v in n]
    cell = torch.arange(math.prod(n), device=DEV)
    ijk, rest = [], cell
    for d in range(dim):
        ijk.append(rest % n[d])
        rest = rest // n[d]
    gid = torch.zeros((len(cell), len(nodes)), dtype=torch.int64, device=DEV)
    stride = 1
    for d in range(dim):
        gid += stride * (order * ijk[d][:, None] + torch.tensor([a[d] for a in nodes], device=DEV)[None, :])
        stride *= fine[d]
    total = stride
    fixed = torch.zeros(total, dtype=torch.bool, device=DEV)
    co, rest = [], torch.arange(total, device=DEV)
    for d in range(dim):
        co.append(rest % fine[d])
        rest = rest // fine[d]
    if bc == "x0":
        fixed = co[0] == 0
    else:
        for d in range(dim):
            fixed |= (co[d] == 0) | (co[d] == fine[d] - 1)
    gid = torch.cat([gid + c * total for c in range(ncomp)], dim=1)
    fixed = fixed.repeat(ncomp)
    pos = (cell[:, None] * len(seq) + rank[None, :]).reshape(-1)
    first = torch.full((total * ncomp,), 1 << 62, dtype=torch.int64, device=DEV)
    first.scatter_reduce_(0, gid.reshape(-1), pos, "amin")
    free = torch.nonzero(~fixed).reshape(-1)
    order_ = torch.argsort(first[free])
    row = torch.full((total * ncomp,), -1, dtype=torch.int64, device=DEV)
    row[free[order_]] = torch.arange(len(free), device=DEV)
    return row[gid], len(free)


def _pcg(apply, diag, b, tol=1e-14, most=20000):
    """Jacobi-PCG in 64 bits, restarted on the true residual until that stops falling."""
    x = torch.zeros_like(b)
    bn = float(b.norm())
    best, kept = math.inf, x
    for _ in range(4):
        r = b - apply(x)
        rn = float(r.norm())
        if rn < best:
            best, kept = rn, x.clone()
        if not rn > tol * bn or (rn > 0.3 * best and rn != best):
            break
        z = r / diag
        p, rz = z.clone(), torch.dot(r, z)
        goal = max(1e-12 * rn, 1e-15 * bn)
        for i in range(most):
            q = apply(p)
            a = rz / torch.dot(p, q)
            x = x + a * p
            r = r - a * q
            if i % 16 == 15 and float(r.norm()) <= goal:
                break
            z = r / diag
            new = torch.dot(r, z)
            p = z + (new / rz) * p
            rz = new
    r = b - apply(x)
    return x if float(r.norm()) < best else kept


def _owners(rows, n):
    """For every row the positions of its DOF in the flattened (cells, nd) array, padded with one past the end."""
    flat = rows.reshape(-1)
    at = torch.nonzero(flat >= 0).reshape(-1)
    r, by = torch.sort(flat[at], stable=True)
    first = torch.searchsorted(r, torch.arange(n, device=DEV))
    rank = torch.arange(len(r), device=DEV) - first[r]
    pos = torch.full((n, int(rank.max()) + 1), len(flat), dtype=torch.int64, device=DEV)
    pos[r, rank] = at[by]
    return pos


def _scatter(pos, ye):
    """Sum of element vectors ye (cells, nd) at their rows (`pos` from _owners)."""
    return torch.cat([ye.reshape(-1), ye.new_zeros(1)])[pos].sum(1)


def _points(n, xi):
    """Quadrature points of every cell of the unit box, (cells, points, dim) as numpy, x fastest."""
    ijk = np.stack([g.transpose().ravel() for g in np.meshgrid(*[np.arange(k) for k in n], indexing="ij")], axis=1)
    return (ijk[:, None, :] + 0.5 * (xi[None, :, :] + 1.0)) / np.array(n)


def _poisson_exact(case, seed):
    n, p = _cells(case), case["order"]
    dim, m = len(n), p + 1
    d = _data(case, seed)
    S, G, W, xi = _shape_tables(dim, p, m)
    rows, nrow = _numbering(n, p, 1, case["bc"])
    cells, nd, nq = math.prod(n), S.shape[0], len(W)
    k = f = None   # (cells, nq) or (1, nq)
    if case["k"] == "const":
        k = torch.full((1, nq), d["k0"], dtype=torch.float64, device=DEV)
    elif case["k"] == "cell":
        k = _t(d["k_cell"])[:, None].expand(cells, nq)
    elif case["k"] == "qpoint":
        xq = _points(n, xi)
        k, f = _t(d["k_fn"](xq)), _t(d["f_fn"](xq))
    else:
        ax = [torch.sin(2 * math.pi * (torch.arange(v, device=DEV, dtype=torch.float64)[:, None]
                                       + _t(0.5 * (_gauss(m)[0] + 1.0))[None, :]) / v) for v in n]   # (layers, points)
        s = ax[0][None, None, :, None, None, :] if dim == 3 else ax[0][None, :, None, :]
        if dim == 3:
            s = s * ax[1][None, :, None, None, :, None] * ax[2][:, None, None, :, None, None]
        else:
            s = s * ax[1][:, None, :, None]
        k = (1.0 + 0.5 * s).reshape(cells, nq)
    if f is None:
        f = torch.full((1, nq), d["f0"], dtype=torch.float64, device=DEV)
    if case["kind"] == "mapped":   # gradients and weights of every cell's own trilinear map
        Sg, Gg, _, _ = _shape_tables(dim, 1, m)
        v = _t(d["vertices"])
        vid = torch.zeros((cells, 1 << dim), dtype=torch.int64, device=DEV)
        stride, rest = 1, torch.arange(cells, device=DEV)
        for e in range(dim):
            vid += stride * ((rest % n[e])[:, None] + torch.tensor([(a >> e) & 1 for a in range(1 << dim)], device=DEV))
            rest = rest // n[e]
            stride *= n[e] + 1
        J = torch.einsum("cai,aqj->cqij", v[vid], _t(Gg))          # dx_i / dxi_j
        inv = torch.linalg.inv(J)
        wq = torch.abs(torch.linalg.det(J)) * _t(W)
        Ke = torch.zeros((cells, nd, nd), dtype=torch.float64, device=DEV)
        for q in range(nq):
            g = (_t(G[:, q])[None, :, :, None] * inv[:, q][:, None, :, :]).sum(2)   # (cells, nd, dim)
            Ke += (k[:, q] * wq[:, q])[:, None, None] * (g[:, :, None, :] * g[:, None, :, :]).sum(3)
        fe = (f * wq) @ _t(S).T
    else:
        h = 1.0 / np.array(n)
        Gp = _t(G * (2.0 / h))                                       # physical gradients
        w = _t(W * np.prod(h / 2.0))
        fe = ((f * w) @ _t(S).T).expand(cells, nd)
        M = torch.einsum("aqd,bqd->qab", Gp, Gp) * w[:, None, None]
        Ke = (k.expand(cells, nq) @ M.reshape(nq, nd * nd)).reshape(cells, nd, nd) if p == 1 else None
    pos = _owners(rows, nrow)
    b = _scatter(pos, fe)
    if p == 1:   # 27-point (9-point) stencil over the vertex grid
        g = [v + 1 for v in n]
        st = torch.zeros([3 ** dim] + list(reversed(g)), dtype=torch.float64, device=DEV)
        for a in range(nd):
            for c in range(nd):
                code, sl = 0, []
                for e in range(dim):
                    code += 3 ** e * (((c >> e) & 1) - ((a >> e) & 1) + 1)
                    sl.insert(0, slice((a >> e) & 1, ((a >> e) & 1) + n[e]))
                st[tuple([code] + sl)] += Ke[:, a, c].reshape(list(reversed(n)))
        del Ke
        vrow = torch.full((math.prod(g),), -1, dtype=torch.int64, device=DEV)   # row of every vertex
        stride, rest = 1, torch.arange(cells, device=DEV)
        vid = torch.zeros((cells, nd), dtype=torch.int64, device=DEV)
        for e in range(dim):
            vid += stride * ((rest % n[e])[:, None] + torch.tensor([(a >> e) & 1 for a in range(nd)], device=DEV))
            rest = rest // n[e]
            stride *= g[e]
        vrow[vid.reshape(-1)] = rows.reshape(-1)
        free = torch.nonzero(vrow >= 0).reshape(-1)
        keep = (vrow >= 0).reshape(list(reversed(g))).to(torch.float64)
        pad = torch.zeros([v + 2 for v in reversed(g)], dtype=torch.float64, device=DEV)
        core = tuple(slice(1, v + 1) for v in reversed(g))

        def apply(x):
            pad[core] = x
            y = torch.zeros_like(keep)
            for code in range(3 ** dim):
                o = [(code // 3 ** e) % 3 for e in range(dim)]
                y.addcmul_(st[code], pad[tuple(slice(o[e], o[e] + g[e]) for e in reversed(range(dim)))])
            return y * keep

        bg = torch.zeros(math.prod(g), dtype=torch.float64, device=DEV)
        bg[free] = b[vrow[free]]
        diag = torch.where(keep > 0, st[(3 ** dim) // 2], torch.ones_like(keep))
        u = _grid_pcg(apply, diag, bg.reshape(keep.shape))
        x = torch.empty(nrow, dtype=torch.float64, device=DEV)
        x[vrow[free]] = u.reshape(-1)[free]
        return x.cpu().numpy()
    T = Gp.reshape(nd, nq * dim)
    kw = (k * w).repeat_interleave(dim, dim=1)
    spare = torch.where(rows < 0, nrow, rows)

    def apply(x):
        xe = torch.cat([x, x.new_zeros(1)])[spare]
        return _scatter(pos, ((xe @ T) * kw) @ T.T)

    diag = _scatter(pos, (kw @ (T * T).T).expand(cells, nd))
    return _pcg(apply, diag, b).cpu().numpy()


def _grid_pcg(apply, diag, b):
    shape = b.shape
    x = _pcg(lambda v: apply(v.reshape(shape)).reshape(-1), diag.reshape(-1), b.reshape(-1))
    return x.reshape(shape)


def _elastic_tables(h, E, nu, body):
    """24 x 24 element matrix and vector of lambda div div + 2 mu eps : eps on a box cell of sides h."""
    S, G, W, _ = _shape_tables(3, 1, 2)
    G = G * (2.0 / np.array(h))
    w = W * np.prod(np.array(h) / 2.0)
    lam, mu = nu * E / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
    K = np.zeros((3, 8, 3, 8))
    for i in range(3):
        for j in range(3):
            K[i, :, j, :] += lam * np.einsum("aq,bq,q->ab", G[:, :, i], G[:, :, j], w)
            K[i, :, j, :] += mu * np.einsum("aq,bq,q->ab", G[:, :, j], G[:, :, i], w)
            if i == j:
                K[i, :, j, :] += mu * np.einsum("aqd,bqd,q->ab", G, G, w)
    fe = np.concatenate([body[i] * (S @ w) for i in range(3)])
    return K.reshape(24, 24), fe


def _constant_exact(rows, nrow, K, fe):
    """Solve of an operator whose cells all have the element matrix K."""
    Kt, spare, pos = _t(K), torch.where(rows < 0, nrow, rows), _owners(rows, nrow)
    cells, nd = rows.shape
    b = _scatter(pos, _t(fe)[None, :].expand(cells, nd))
    diag = _scatter(pos, torch.diagonal(Kt)[None, :].expand(cells, nd))
    return _pcg(lambda x: _scatter(pos, torch.cat([x, x.new_zeros(1)])[spare] @ Kt.T), diag, b)


def _serve_exact(n, E, nu):
    K, fe = _elastic_tables((1.0 / n,) * 3, E, nu, (0.0, 0.0, -1.0))
    cell = torch.arange(n ** 3, device=DEV)
    i, j, k = cell % n, (cell // n) % n, cell // (n * n)
    cols = []
    for l in range(24):
        c, a = divmod(l, 8)
        x, y, z = i + (a & 1), j + ((a >> 1) & 1), k + (a >> 2)
        cols.append(torch.where(x > 0, 3 * ((x - 1) + n * (y + (n + 1) * z)) + c, -1))
    return _constant_exact(torch.stack(cols, dim=1), 3 * n * (n + 1) ** 2, K, fe).cpu().numpy()


def _batch_exact(dim, n, k, f0):
    """On the uniform mesh the Gauss-integrated load of prod sin(pi x) is itself a discrete sine mode, an
    eigenvector of the stiffness and mass stencils, so the solution is that mode scaled."""
    h = 1.0 / n
    x = np.arange(1, n) * h
    load = 0.0   # load stencil of sin(pi x): sum over the two cells of the two Gauss points
    gx, gw = _gauss(2)
    for xi, w in zip(gx, gw):
        t = 0.5 * (xi + 1.0)
        load += 0.5 * h * w * (t * math.cos(math.pi * h * (t - 1.0)) + (1.0 - t) * math.cos(math.pi * h * t))
    c = math.cos(math.pi * h)
    stiff, mass = 4.0 * math.sin(0.5 * math.pi * h) ** 2 / h, h * (4.0 + 2.0 * c) / 6.0
    amp = f0 * dim * math.pi ** 2 * load ** dim / (dim * stiff * mass ** (dim - 1))
    s = np.sin(math.pi * x)
    u = s
    for _ in range(dim - 1):
        u = np.multiply.outer(s, u)
    return amp * u.ravel()


def _multifield_exact(case, seed):
    n = case["n"]
    kappa, sigma, f = _two_fields(seed)
    h = 1.0 / n
    rows, sizes, tabs = [], [], []
    for order in (2, 1):
        r, m = _numbering((n, n, n), order, 1, "boundary")
        rows.append(r)
        sizes.append(m)
        tabs.append(_shape_tables(3, order, 3))
    W = tabs[0][2] * (h / 2.0) ** 3
    nd = [27, 8]
    K = np.zeros((35, 35))
    fe = np.zeros(35)
    at = [slice(0, 27), slice(27, 35)]
    for a in range(2):
        G = tabs[a][1] * (2.0 / h)
        fe[at[a]] = f[a] * (tabs[a][0] @ W)
        for b in range(2):
            mass = np.einsum("aq,bq,q->ab", tabs[a][0], tabs[b][0], W)
            K[at[a], at[b]] += sigma * mass if a == b else -sigma * mass
            if a == b:
                K[at[a], at[b]] += kappa[a] * np.einsum("aqd,bqd,q->ab", G, G, W)
    both = torch.cat([rows[0], torch.where(rows[1] < 0, -1, rows[1] + sizes[0])], dim=1)
    return _constant_exact(both, sum(sizes), K, fe).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("poisson", "new_mesh", "mapped"):
        return _poisson_exact(case, seed)
    if kind == "elasticity":
        n = _cells(case)
        E, nu, body = _elastic(seed)
        K, fe = _elastic_tables([1.0 / v for v in n], E, nu, body)
        rows, nrow = _numbering(n, 1, 3, "x0")
        return _constant_exact(rows, nrow, K, fe).cpu().numpy()
    if kind == "multifield":
        return _multifield_exact(case, seed)
    if kind == "batch":
        return np.concatenate([_batch_exact(*p) for p in _batch_problems(case, seed)])
    return [_serve_exact(*r) for r in _serve_requests(case, seed)]
