"""Which boxes are solved from the cells and which on the stored matrix
(lattice_pays of cg.hip): boxes of sides near one size and short wide ones from
the cells, long ones of small cross-section, whose march would leave the chip idle,
on the stored matrix; a solver changes over when its operator's coefficient does.
The route shows in the bytes of femhip_solver_profile_spmv; solutions against the
oracle (unit cells, so that a long box is no worse conditioned than a wide one)."""
import numpy as np
import pytest

import fempar_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # n, order, k, bc, from the cells
    ((66, 67), 1, "sin3", "boundary", True),
    ((3000, 4), 1, "const", "boundary", True),
    ((4, 6000), 1, "const", "boundary", False),
    ((33, 34), 2, "const", "boundary", True),
    ((1, 9000), 2, "cell", "boundary", False),
    ((18, 19, 17), 1, "cell", "x0", True),
    ((3, 3, 5000), 1, "sin3", "boundary", False),
    ((9, 10, 11), 2, "sin3", "boundary", True),
    ((1, 1, 3000), 2, "const", "boundary", False),
    ((11, 9, 10), 1, "elasticity", "x0", True),
    ((1, 1, 5000), 1, "elasticity", "x0", False),
]


def _k(x):
    return 1.0 + 0.4 * np.sin(x[..., 0]) * np.cos(3 * x[..., 1])


def _build(env, n, order, k, bc):
    dim = len(n)
    lim = [v for a in n for v in (0, a)]
    kc = np.exp(np.random.default_rng(3).normal(0.0, 0.5, int(np.prod(n)))) if k == "cell" else None
    ncomp = 3 if k == "elasticity" else 1
    osp = O.Space(O.make_problem(dim, n, order, ncomp, {"boundary": O.BC_ALL, "x0": O.BC_X0}[bc], lim=lim + [0, 0] * (3 - dim)))
    tria = F.serial_triangulation_t().create(env, {
        "STRUCT_HEX_MESH_GENERATOR_NUM_DIMS": dim, "STRUCT_HEX_MESH_GENERATOR_NUM_CELLS_X_DIM": list(n),
        "STRUCT_HEX_MESH_GENERATOR_DOMAIN_LIMITS": lim})
    fes = F.serial_fe_space_t().create(tria, order=order, num_components=ncomp, dirichlet=bc)
    if k == "elasticity":
        oph = O.make_physics(kind=O.PHYS_ELASTICITY, E=20.0, nu=0.35, body=(0.5, 0.0, -1.0))
        di = F.linear_elasticity_discrete_integration_t(20.0, 0.35, (0.5, 0.0, -1.0))
    else:
        oph = O.make_physics(k_kind={"const": O.K_CONST, "sin3": O.K_SIN3, "cell": O.K_CELL}[k], k0=1.5, k_cell=kc,
                             f_kind=O.F_CONST, f0=2.0)
        di = F.poisson_discrete_integration_t(k=k, k0=1.5, k_cell=kc, f="const", f0=2.0)
    op = F.fe_affine_operator_t()
    op.create("CSR", [True], fes, di)
    op.compute()
    return osp, oph, op


def _solver(env, op, precision, rtol):
    s = F.iterative_linear_solver_t().create(env)
    s.set_type_from_string("CG")
    s.set_parameters_from_pl({"ILS_RTOL": rtol, "ILS_MAX_NUM_ITERATIONS": 20000, "FEMHIP_PRECISION": precision})
    s.set_operators(op, F.jacobi_preconditioner_t(op))
    return s


def _from_cells(s, op, precision, values):
    """One-launch passes: vectors in and out, S or M, and the coefficient's values a cell."""
    nbytes = s.profile_spmv(1)[1]
    return nbytes == op.n * ((32.0 if precision == "FP32_REFINED" else 64.0) + 8.0) + 8.0 * values


@pytest.mark.parametrize("n,order,k,bc,cells", CASES)
def test_route_and_solution(env, n, order, k, bc, cells):
    print(f"[route] {n} Q{order} {k} {bc}", flush=True)
    osp, oph, op = _build(env, n, order, k, bc)
    irp, ja, val, rhs = osp.assemble(oph, True)
    ref, info = O.cg(irp, ja, val, rhs, True, precond="jacobi", rtol=1e-12, maxit=20000)
    assert info["converged"]
    for precision, rtol, tol in (("FP64", 1e-12, 1e-9), ("FP32_REFINED", 1e-10, 1e-7)):
        s = _solver(env, op, precision, rtol)
        x = s.solve()
        assert s.did_converge() and np.linalg.norm(x - ref) <= tol * np.linalg.norm(ref), precision
        assert _from_cells(s, op, precision, np.prod(n) if k == "cell" else 0) == cells, precision


def test_route_follows_the_coefficient(env):
    """A flat box of Q2 cells: from the cells with a constant, on the stored matrix with
    point values, back again; one solver, each solution that of its operator's rows."""
    n = (4, 5, 33)
    _, _, op = _build(env, n, 2, "const", "x0")
    s = _solver(env, op, "FP32_REFINED", 1e-10)
    fes = op.fe_space
    for di, cells in ((F.poisson_discrete_integration_t(k="const", k0=1.5, f="const", f0=2.0), True),
                      (F.poisson_discrete_integration_t(k=_k, f=lambda x: 1.0 + x[..., 0]), False),
                      (F.poisson_discrete_integration_t(k="const", k0=0.3, f="const", f0=1.0), True)):
        op.discrete_integration = di
        op._phys = di.physics(fes)
        F._native.check(op._lib.femhip_operator_set_physics(op.h, op._phys))
        op.compute()
        A, rhs = op.get_matrix(), op.get_translation()
        x = s.solve()
        ref, _ = O.cg(A.irp, A.ja, A.val, rhs, True, precond="jacobi", rtol=1e-12, maxit=20000)
        assert s.did_converge() and np.linalg.norm(x - ref) <= 1e-7 * np.linalg.norm(ref)
        assert np.array_equal(s.get_solution(), x)
        assert _from_cells(s, op, "FP32_REFINED", 0) == cells
