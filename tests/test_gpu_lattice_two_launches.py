"""Iterations in two launches (k_lat_a and k_lat_b, k_lat_rf_a and k_lat_rf_b of
cg_lattice.h) on systems just above the sizes where they begin: 3,000,000 rows,
or 1,000,000 of 3-D Q2 and of elasticity.  2-D and 3-D, Q1 and Q2, every kind of
coefficient, both boundary kinds, both preconditioners, every remainder of the
rows by 4 (the vector kernels load two or four rows at a time).

References use the operator's assembled rows (held to the oracle's at other
sizes) and the oracle's product.  The first iterations are cg.f90's with pairwise
sums: an early iterate is fixed to about 1e-15 times the iterations, so it is held
to 1e-10.  (The oracle's own sums run from the first row to the last: over three
million equal terms they round by 3e-11, and its fifth iterate is 2.3e-10 from
the one with long double sums; pairwise sums leave 2.6e-13.)  Converged solutions
are held by their residual: rtol of the first one, and for each product the
rounding of up to 125 terms a row."""
import numpy as np
import pytest

import fempar_amd as F
from oracle import oracle as O
from test_gpu_lattice import _f, _k
from test_lattice_plan import plan

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
CASES = [
    # n, order, k, bc, precond
    ((145, 145, 146), 1, "sin3", "boundary", "jacobi"),
    ((146, 146, 146), 1, "cell", "boundary", "identity"),
    ((144, 143, 144), 1, "qpoint", "x0", "jacobi"),
    ((1734, 1734), 1, "cell", "x0", "jacobi"),
    ((867, 868), 2, "qpoint", "boundary", "jacobi"),
    ((50, 51, 51), 2, "sin3", "boundary", "jacobi"),
    ((51, 49, 50), 2, "cell", "x0", "identity"),
    ((50, 50, 52), 2, "qpoint", "boundary", "jacobi"),
    ((69, 70, 70), 1, "elasticity", "x0", "jacobi"),
]


def _operator(env, n, order, k, bc):
    dim = len(n)
    elastic = k == "elasticity"
    assert not plan(n, order, 3 if elastic else 1, F._native.BC_ALL_BOUNDARY if bc == "boundary" else F._native.BC_X0_FACE).one
    tria = F.serial_triangulation_t().create(env, {
        "STRUCT_HEX_MESH_GENERATOR_NUM_DIMS": dim, "STRUCT_HEX_MESH_GENERATOR_NUM_CELLS_X_DIM": list(n),
        "STRUCT_HEX_MESH_GENERATOR_DOMAIN_LIMITS": [0, 1, -0.5, 1, 0, 2][: 2 * dim]})
    fes = F.serial_fe_space_t().create(tria, order=order, num_components=3 if elastic else 1, dirichlet=bc)
    if elastic:
        di = F.linear_elasticity_discrete_integration_t(20.0, 0.35, (0.5, 0.0, -1.0))
    elif k == "qpoint":
        di = F.poisson_discrete_integration_t(k=_k, f=_f)
    else:
        kc = np.exp(np.random.default_rng(3).normal(0.0, 0.5, int(np.prod(n)))) if k == "cell" else None
        di = F.poisson_discrete_integration_t(k=k, k0=1.5, k_cell=kc, f="const", f0=2.0)
    op = F.fe_affine_operator_t()
    op.create("CSR", [True], fes, di)
    op.compute()
    return op


def _solver(env, op, precond, **params):
    s = F.iterative_linear_solver_t().create(env)
    s.set_type_from_string("CG")
    s.set_parameters_from_pl(params)
    s.set_operators(op, F.jacobi_preconditioner_t(op) if precond == "jacobi" else F.identity_operator_t(op))
    return s


def _iterates(A, b, x0, precond, its):
    """cg.f90:101-238: the last iterate and ||r|| after each."""
    M = 1.0 / O.extract_diagonal(A.irp, A.ja, A.val) if precond == "jacobi" else np.ones(len(b))
    x = np.zeros(len(b)) if x0 is None else x0.copy()
    r = b - O.spmv(A.irp, A.ja, A.val, x, True)
    p = M * r
    rz, hist = r @ p, []
    for _ in range(its):
        q = O.spmv(A.irp, A.ja, A.val, p, True)
        alpha = rz / (p @ q)
        x += alpha * p
        r -= alpha * q
        hist.append(np.sqrt(r @ r))
        z = M * r
        rz, last = r @ z, rz
        p = z + (rz / last) * p
    return x, np.array(hist)


@pytest.mark.parametrize("n,order,k,bc,precond", CASES)
def test_two_launch_solves(env, n, order, k, bc, precond):
    op = _operator(env, n, order, k, bc)
    print(f"[two launches] {n} Q{order} {k} {bc} {precond}: {op.n} rows", flush=True)
    A = op.get_matrix()
    rng = np.random.default_rng(11)
    b, x0 = rng.standard_normal(op.n), rng.standard_normal(op.n)
    # iteration limit: the iterate itself, from a right-hand side and a guess and from the operator's own
    for its, rhs, guess in ((1, b, x0), (16, b, x0), (5, None, None)):
        s = _solver(env, op, precond, ILS_RTOL=1e-14, ILS_MAX_NUM_ITERATIONS=its)
        x = s.solve(rhs, guess)
        assert not s.did_converge() and s.get_num_iterations() == its
        ref, norms = _iterates(A, op.get_translation() if rhs is None else rhs, guess, precond, its)
        assert np.linalg.norm(x - ref) <= 1e-10 * np.linalg.norm(ref), its
        hist = s.get_error_estimate_history_convergence_test()
        assert len(hist) == its and np.max(np.abs(hist / norms - 1.0)) <= 1e-7
        if its == 16:   # FP32 vectors: 16 steps of a few roundings of 6e-8, each carried through the others
            s = _solver(env, op, precond, ILS_RTOL=1e-14, ILS_MAX_NUM_ITERATIONS=its, FEMHIP_PRECISION="FP32_REFINED")
            x = s.solve(rhs, guess)
            assert not s.did_converge() and s.get_num_iterations() == its
            assert np.linalg.norm(x - ref) <= 16 * 16 * 4 * 6e-8 * np.linalg.norm(ref)
    # convergence
    r0 = np.linalg.norm(b - O.spmv(A.irp, A.ja, A.val, x0, True))
    for precision, rtol in (("FP64", 1e-7), ("FP32_REFINED", 1e-7)):
        s = _solver(env, op, precond, ILS_RTOL=rtol, ILS_MAX_NUM_ITERATIONS=20000, FEMHIP_PRECISION=precision)
        x = s.solve(b, x0)
        assert s.did_converge() and 16 < s.get_num_iterations() < 20000, precision
        rn = np.linalg.norm(b - O.spmv(A.irp, A.ja, A.val, x, True))
        rounding = 125 * EPS * np.linalg.norm(O.spmv(A.irp, A.ja, np.abs(A.val), np.abs(x), True))
        assert abs(s.result["true_residual"] - rn) <= rounding, precision
        # FP64 stops by the recurrence's residual, which leaves the true one by a rounding an iteration
        gap = rounding * (np.sqrt(s.get_num_iterations()) if precision == "FP64" else 1.0)
        assert rn <= rtol * r0 * (1.0 + 1e-6) + gap, precision
    op.free()


@pytest.fixture(scope="module")
def criteria_operator(env):
    op = _operator(env, (1734, 1735), 1, "sin3", "boundary")
    A = op.get_matrix()
    yield op, A
    op.free()


@pytest.mark.parametrize("crit", O.CRITERIA)
def test_two_launch_stopping_criteria(env, criteria_operator, crit):
    """As test_gpu_parity's: the count, the threshold and every estimate of the
    history; no estimate lies within 1 % of its threshold."""
    op, A = criteria_operator
    print(f"[two launches] {crit}", flush=True)
    b = np.random.default_rng(11).standard_normal(op.n)
    rtol = 0.8 if crit.startswith("DELTA_DELTA") else 0.3
    ref, info = O.cg(A.irp, A.ja, A.val, b, True, precond="jacobi", criterion=crit, rtol=rtol, maxit=30, history=True)
    assert info["converged"] and np.all(np.abs(info["history"] / info["rhs_test"] - 1.0) > 0.01)
    s = _solver(env, op, "jacobi", ILS_RTOL=rtol, ILS_MAX_NUM_ITERATIONS=30, ILS_STOPPING_CRITERIUM=crit)
    x = s.solve(b)
    assert s.did_converge() and s.get_num_iterations() == info["iterations"]
    assert abs(s.result["rhs_convergence_test"] - info["rhs_test"]) <= 1e-9 * info["rhs_test"]
    hist = s.get_error_estimate_history_convergence_test()
    assert len(hist) == info["iterations"] and np.max(np.abs(hist / info["history"] - 1.0)) <= 1e-7
    assert np.linalg.norm(x - ref) <= 1e-10 * np.linalg.norm(ref)
