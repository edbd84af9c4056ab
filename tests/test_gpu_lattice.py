"""Products formed from the cells (lattice.h) against the oracle.

Sizes at the edges of the workgroup tiles and chunks (one cell more or less
than a tile, thin and long boxes, a single layer), 2-D and 3-D, Q1 and Q2, one
coefficient a cell, the closed form and point values, the two Dirichlet kinds
(the free nodes' box with and without its last planes) and both preconditioners,
with iterations in one launch (in two: test_gpu_lattice_two_launches.py).

Gates: FP64 solutions to 1e-12 within 1e-10 relative of the oracle's, in no more
than 2 % + 2 of its iterations; FP32-refined within 1e-8 (the gates of test_gpu_parity)."""
import numpy as np
import pytest

import fempar_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # n, order, k, bc, precond
    ((65, 66), 1, "sin3", "boundary", "jacobi"),
    ((300, 17), 1, "cell", "x0", "jacobi"),
    ((600, 9), 1, "const", "boundary", "jacobi"),
    ((70, 64), 1, "qpoint", "x0", "identity"),
    ((33, 40), 2, "sin3", "x0", "jacobi"),
    ((130, 9), 2, "qpoint", "boundary", "jacobi"),
    ((17, 18, 19), 1, "sin3", "boundary", "jacobi"),
    ((64, 9, 12), 1, "cell", "x0", "identity"),
    ((2, 60, 70), 1, "const", "x0", "jacobi"),
    ((45, 45, 4), 1, "qpoint", "boundary", "jacobi"),
    ((600, 4, 5), 1, "sin3", "x0", "jacobi"),
    ((9, 10, 11), 2, "sin3", "boundary", "jacobi"),
    ((65, 3, 4), 2, "cell", "x0", "jacobi"),
    ((4, 5, 33), 2, "qpoint", "x0", "identity"),
    ((1, 24, 30), 2, "const", "x0", "jacobi"),
]


def _k(x):
    return 1.0 + 0.4 * np.sin(2 * np.pi * x[..., 0]) * np.cos(3 * x[..., 1]) + (0.2 * x[..., 2] if x.shape[-1] == 3 else 0.0)


def _f(x):
    return 1.0 + x[..., 0] - 2.0 * x[..., 1] ** 2


def _build(env, n, order, k, bc):
    dim = len(n)
    lim = [0, 1, -0.5, 1, 0, 2][: 2 * dim]
    kc = np.exp(np.random.default_rng(3).normal(0.0, 1.0, int(np.prod(n)))) if k == "cell" else None
    osp = O.Space(O.make_problem(dim, n, order, 1, {"boundary": O.BC_ALL, "x0": O.BC_X0}[bc], lim=lim + [0, 0] * (3 - dim)))
    tria = F.serial_triangulation_t().create(env, {
        "STRUCT_HEX_MESH_GENERATOR_NUM_DIMS": dim, "STRUCT_HEX_MESH_GENERATOR_NUM_CELLS_X_DIM": list(n),
        "STRUCT_HEX_MESH_GENERATOR_DOMAIN_LIMITS": lim})
    fes = F.serial_fe_space_t().create(tria, order=order, dirichlet=bc)
    if k == "qpoint":
        xq = fes.get_quadrature_points_coordinates()
        oph = O.make_physics(k_kind=O.K_QPOINT, k_qp=_k(xq).reshape(-1), f_kind=O.F_QPOINT, f_qp=_f(xq).reshape(-1))
        di = F.poisson_discrete_integration_t(k=_k, f=_f)
    else:
        oph = O.make_physics(k_kind={"const": O.K_CONST, "sin3": O.K_SIN3, "cell": O.K_CELL}[k], k0=1.5, k_cell=kc,
                             f_kind=O.F_CONST, f0=2.0)
        di = F.poisson_discrete_integration_t(k=k, k0=1.5, k_cell=kc, f="const", f0=2.0)
    op = F.fe_affine_operator_t()
    op.create("CSR", [True], fes, di)
    return osp, oph, op


def _solve(env, op, precision, precond, rtol, b=None, x=None):
    s = F.iterative_linear_solver_t().create(env)
    s.set_type_from_string("CG")
    s.set_parameters_from_pl({"ILS_RTOL": rtol, "ILS_MAX_NUM_ITERATIONS": 20000, "FEMHIP_PRECISION": precision})
    s.set_operators(op, F.jacobi_preconditioner_t(op) if precond == "jacobi" else F.identity_operator_t(op))
    return s, s.solve(b, x)


@pytest.mark.parametrize("n,order,k,bc,precond", CASES)
def test_lattice_solves_match_oracle(env, n, order, k, bc, precond):
    print(f"[lattice] {n} Q{order} {k} {bc} {precond}", flush=True)
    osp, oph, op = _build(env, n, order, k, bc)
    op.compute()
    irp, ja, val, rhs = osp.assemble(oph, True)
    assert len(rhs) == op.n > 4096
    ref, info = O.cg(irp, ja, val, rhs, True, precond=precond, rtol=1e-12, maxit=20000)
    s, x = _solve(env, op, "FP64", precond, 1e-12)
    # rounding alone moves the count of long solves (64 x 9 x 12 without Jacobi: 1194 to
    # 1210 for the same matrix by the order of the sums), so it is only held not to grow
    assert s.did_converge() and s.get_num_iterations() <= 1.02 * info["iterations"] + 2
    assert np.linalg.norm(x - ref) <= 1e-10 * np.linalg.norm(ref)
    # the reported residual: both sums round each of up to 125 products a row
    r = rhs - O.spmv(irp, ja, val, x, True)
    bound = 125 * np.finfo(float).eps * np.linalg.norm(O.spmv(irp, ja, np.abs(val), np.abs(x), True))
    assert abs(s.result["true_residual"] - np.linalg.norm(r)) <= bound
    s, x = _solve(env, op, "FP32_REFINED", precond, 1e-10)
    assert s.did_converge() and np.linalg.norm(x - ref) <= 1e-8 * np.linalg.norm(ref)
    # another right-hand side and a first guess, in the operator's row order
    rng = np.random.default_rng(11)
    b, x0 = rng.standard_normal(op.n), rng.standard_normal(op.n)
    ref, _ = O.cg(irp, ja, val, b, True, precond=precond, rtol=1e-12, maxit=20000)
    for precision, rtol, tol in (("FP64", 1e-12, 1e-9), ("FP32_REFINED", 1e-10, 1e-7)):
        s, x = _solve(env, op, precision, precond, rtol, b, x0)
        assert s.did_converge() and np.linalg.norm(x - ref) <= tol * np.linalg.norm(ref), precision


@pytest.mark.parametrize("n", [(9, 13, 11), (2, 30, 30), (33, 9, 8)])
def test_lattice_elasticity_matches_oracle(env, n):
    """Vector Q1 elasticity on the lattice: component-blocked rows inside, the
    operator's first-touch order outside (right-hand side, guess and solution)."""
    print(f"[lattice] elasticity {n}", flush=True)
    lim = [0, 1, -0.5, 1, 0, 2]
    osp = O.Space(O.make_problem(3, n, 1, 3, O.BC_X0, lim=lim))
    irp, ja, val, rhs = osp.assemble(O.make_physics(kind=O.PHYS_ELASTICITY, E=20.0, nu=0.35, body=(0.5, 0.0, -1.0)), True)
    tria = F.serial_triangulation_t().create(env, {
        "STRUCT_HEX_MESH_GENERATOR_NUM_DIMS": 3, "STRUCT_HEX_MESH_GENERATOR_NUM_CELLS_X_DIM": list(n),
        "STRUCT_HEX_MESH_GENERATOR_DOMAIN_LIMITS": lim})
    fes = F.serial_fe_space_t().create(tria, order=1, num_components=3, dirichlet="x0")
    op = F.fe_affine_operator_t()
    op.create("CSR", [True], fes, F.linear_elasticity_discrete_integration_t(20.0, 0.35, (0.5, 0.0, -1.0)))
    op.compute()
    assert op.n == len(rhs) > 4096
    rng = np.random.default_rng(5)
    b, x0 = rng.standard_normal(op.n), rng.standard_normal(op.n)
    for rh, guess in ((rhs, None), (b, x0)):
        ref, info = O.cg(irp, ja, val, rh, True, precond="jacobi", rtol=1e-12, maxit=50000)
        for precision, rtol, tol in (("FP64", 1e-12, 1e-9), ("FP32_REFINED", 1e-10, 1e-7)):
            s, x = _solve(env, op, precision, "jacobi", rtol, None if rh is rhs else rh, guess)
            assert s.did_converge() and np.linalg.norm(x - ref) <= tol * np.linalg.norm(ref), precision


def test_lattice_both_forms_and_limits(env):
    """A system of more than 400,000 rows (two launches an iteration) and one of
    fewer give the same solution as their assembled rows; the iteration limit
    and a coefficient set anew hold on the path."""
    for n in ((76, 77, 78), (30, 31, 29)):
        osp, oph, op = _build(env, n, 1, "cell", "boundary")
        op.compute()
        A = op.get_matrix()
        rhs = op.get_translation()
        for precision in ("FP64", "FP32_REFINED"):
            s, x = _solve(env, op, precision, "jacobi", 1e-11)
            assert s.did_converge()
            r = rhs - O.spmv(A.irp, A.ja, A.val, x, True)
            assert np.linalg.norm(r) <= 1.01e-11 * np.linalg.norm(rhs) + 1e-15 * np.linalg.norm(rhs) * max(n)
        for its in (1, 2, 15, 16, 17, 33):
            s = F.iterative_linear_solver_t().create(env)
            s.set_type_from_string("CG")
            s.set_parameters_from_pl({"ILS_RTOL": 1e-14, "ILS_MAX_NUM_ITERATIONS": its})
            s.set_operators(op, F.jacobi_preconditioner_t(op))
            x = s.solve()
            assert not s.did_converge() and s.get_num_iterations() == its
            ref, info = O.cg(A.irp, A.ja, A.val, rhs, True, precond="jacobi", rtol=1e-30, maxit=its)
            assert np.linalg.norm(x - ref) <= 1e-10 * np.linalg.norm(ref), its
    # the same solver after another coefficient: nothing of the first is left
    s, x1 = _solve(env, op, "FP64", "jacobi", 1e-12)
    op.discrete_integration = F.poisson_discrete_integration_t(k="const", k0=0.25, f="const", f0=1.0)
    op._phys = op.discrete_integration.physics(op.fe_space)
    F._native.check(op._lib.femhip_operator_set_physics(op.h, op._phys))
    op.compute()
    x2 = s.solve()
    A, rhs = op.get_matrix(), op.get_translation()
    assert np.linalg.norm(rhs - O.spmv(A.irp, A.ja, A.val, x2, True)) <= 1.01e-12 * np.linalg.norm(rhs) * 10
    # vertices moved afterwards: back to the stored matrix, same solution for the same vertices
    tria = op.fe_space.triangulation
    vc = np.ascontiguousarray(tria.get_uniform_vertex_coordinates())
    F._native.check(op._lib.femhip_space_set_vertex_coords(op.fe_space.h, F._native.ptr(vc)))
    op.compute()
    x3 = s.solve()
    assert s.did_converge() and np.linalg.norm(x3 - x2) <= 1e-10 * np.linalg.norm(x2)


@pytest.mark.parametrize("n,k,bc", [((1, 200, 20), "cell", "boundary"), ((2, 128, 8), "sin3", "boundary"),
                                    ((1, 127, 4), "cell", "x0")])
def test_thin_q2_boxes_match_oracle(env, n, k, bc):
    """Q2 boxes one or two cells thick along x whose tiles are cut short by the
    nodes after them, one a thread: every cell column is solved.  Solutions of a
    matrix half an ulp off differ by 2e-13 at most (direct solves)."""
    print(f"[lattice] thin {n} {k} {bc}", flush=True)
    osp, oph, op = _build(env, n, 2, k, bc)
    op.compute()
    irp, ja, val, rhs = osp.assemble(oph, True)
    assert len(rhs) == op.n > 4096
    ref, _ = O.cg(irp, ja, val, rhs, True, precond="jacobi", rtol=1e-12, maxit=20000)
    bound = 125 * np.finfo(float).eps
    for precision, rtol, tol in (("FP64", 1e-12, 1e-10), ("FP32_REFINED", 1e-10, 1e-8)):
        s, x = _solve(env, op, precision, "jacobi", rtol)
        assert s.did_converge() and np.linalg.norm(x - ref) <= tol * np.linalg.norm(ref), precision
        r = rhs - O.spmv(irp, ja, val, x, True)
        rounding = bound * np.linalg.norm(O.spmv(irp, ja, np.abs(val), np.abs(x), True))
        assert abs(s.result["true_residual"] - np.linalg.norm(r)) <= rounding
