"""CG of small systems in one workgroup (cg_small.h) against the oracle.

Rows around a wave, a workgroup's rows a thread (512 threads, 1 to 8 rows) and
the largest system it takes (4096), both symmetric stencils, the streamed
layouts, stencils too wide for their margins, more iterations than one launch
makes, every stopping criterion and the iteration limit.

Gates as for the other FP64 paths: solutions to 1e-12 within 1e-10 relative of
the oracle's in no more than 2 % + 2 of its iterations."""
import numpy as np
import pytest

import fempar_amd as F
from oracle import oracle as O
from test_gpu_lattice import _build, _solve

pytestmark = pytest.mark.gpu

CASES = [
    # n, order, k, bc, precond
    ((2, 2), 1, "sin3", "boundary", "jacobi"),
    ((9, 9), 1, "cell", "boundary", "jacobi"),
    ((14, 6), 1, "sin3", "boundary", "identity"),
    ((33, 17), 1, "cell", "boundary", "jacobi"),
    ((28, 20), 1, "qpoint", "boundary", "jacobi"),
    ((33, 33), 1, "sin3", "boundary", "jacobi"),
    ((40, 27), 1, "cell", "x0", "jacobi"),
    ((65, 33), 1, "sin3", "boundary", "jacobi"),
    ((65, 65), 1, "cell", "boundary", "jacobi"),
    ((600, 7), 1, "const", "boundary", "jacobi"),
    ((4, 800), 1, "cell", "boundary", "jacobi"),
    ((3, 2, 2), 1, "cell", "boundary", "jacobi"),
    ((9, 9, 9), 1, "sin3", "boundary", "jacobi"),
    ((11, 11, 11), 1, "cell", "boundary", "identity"),
    ((14, 13, 14), 1, "qpoint", "boundary", "jacobi"),
    ((14, 14, 14), 1, "sin3", "boundary", "jacobi"),
    ((12, 15), 2, "cell", "boundary", "jacobi"),
    ((32, 32), 2, "sin3", "boundary", "jacobi"),
    ((4, 5, 4), 2, "cell", "x0", "jacobi"),
    ((8, 8, 8), 2, "const", "boundary", "jacobi"),
]


@pytest.mark.parametrize("n,order,k,bc,precond", CASES)
def test_small_solves_match_oracle(env, n, order, k, bc, precond):
    print(f"[small] {n} Q{order} {k} {bc} {precond}", flush=True)
    osp, oph, op = _build(env, n, order, k, bc)
    op.compute()
    irp, ja, val, rhs = osp.assemble(oph, True)
    assert len(rhs) == op.n <= 4096
    rng = np.random.default_rng(11)
    b, x0 = rng.standard_normal(op.n), rng.standard_normal(op.n)
    for rh, guess, tol in ((rhs, None, 1e-10), (b, x0, 1e-9)):
        ref, info = O.cg(irp, ja, val, rh, True, precond=precond, rtol=1e-12, maxit=20000,
                         **({} if guess is None else {"x0": guess}))
        s, x = _solve(env, op, "FP64", precond, 1e-12, None if rh is rhs else rh, guess)
        assert s.did_converge() and s.get_num_iterations() <= 1.02 * info["iterations"] + 2
        assert np.linalg.norm(x - ref) <= tol * np.linalg.norm(ref)
    # again on the same solver, after other values of the operator
    op.compute()
    x2 = s.solve(b, x0)
    assert np.array_equal(x, x2)


@pytest.mark.parametrize("limit", [1, 7, 1024, 1025])
def test_small_iteration_limit(env, limit):
    """The limit ends the solve where the oracle's ends, inside a launch, at its
    end and in the next one; the history has every iteration."""
    osp, oph, op = _build(env, (600, 7), 1, "const", "boundary")
    op.compute()
    irp, ja, val, rhs = osp.assemble(oph, True)
    _, info = O.cg(irp, ja, val, rhs, True, precond="jacobi", rtol=1e-30, maxit=limit)
    s = F.iterative_linear_solver_t().create(env)
    s.set_type_from_string("CG")
    s.set_parameters_from_pl({"ILS_RTOL": 1e-30, "ILS_MAX_NUM_ITERATIONS": limit})
    s.set_operators(op, F.jacobi_preconditioner_t(op))
    s.solve()
    assert not s.did_converge() and s.get_num_iterations() == info["iterations"] == limit
    h = s.get_error_estimate_history_convergence_test()
    assert len(h) == limit and np.all(h > 0)
