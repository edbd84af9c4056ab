"""The iteration limit of refined solves on a stored FP32 matrix: a reliable update
takes a slot of its own, and those slots are no iterations.  In three kernels a slot
and in two, with the FP32 copy of the matrix and with FP32_STRICT's own."""
import numpy as np
import pytest

import fempar_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SYSTEMS = [("q1", (30, 31, 29), 1, "FP32_REFINED", True), ("q2", (9, 10, 11), 2, "FP32_REFINED", True),
           ("strict", (30, 31, 29), 1, "FP32_STRICT", False), ("few_rows", (15, 16), 1, "FP32_REFINED", False)]


@pytest.mark.parametrize("name,n,order,precision,moved", SYSTEMS, ids=[s[0] for s in SYSTEMS])
def test_refined_limit_on_stored_matrix(env, name, n, order, precision, moved):
    print(f"[refined limit] {name} {precision}", flush=True)
    tria = F.serial_triangulation_t().create(env, {
        "STRUCT_HEX_MESH_GENERATOR_NUM_DIMS": len(n), "STRUCT_HEX_MESH_GENERATOR_NUM_CELLS_X_DIM": list(n),
        "STRUCT_HEX_MESH_GENERATOR_DOMAIN_LIMITS": [0, 1] * len(n)})
    fes = F.serial_fe_space_t().create(tria, order=order)
    if moved:   # vertices given by the caller, though where they were: products from the stored matrix
        vc = np.ascontiguousarray(tria.get_uniform_vertex_coordinates())
        F._native.check(fes._lib.femhip_space_set_vertex_coords(fes.h, F._native.ptr(vc)))
    op = F.fe_affine_operator_t()
    op.create("CSR", [True], fes, F.poisson_discrete_integration_t(k="const", k0=1.5, f="const", f0=2.0))
    op.compute()
    A, rhs = op.get_matrix(), op.get_translation()

    def solve(**params):
        s = F.iterative_linear_solver_t().create(env)
        s.set_type_from_string("CG")
        s.set_parameters_from_pl({"FEMHIP_PRECISION": precision, **params})
        s.set_operators(op, F.jacobi_preconditioner_t(op))
        x = s.solve()
        r = rhs - O.spmv(A.irp, A.ja, A.val, x, True)
        rounding = 125 * np.finfo(float).eps * np.linalg.norm(O.spmv(A.irp, A.ja, np.abs(A.val), np.abs(x), True))
        # the last iterations are in x: its residual is the one the last update found
        assert abs(s.result["error_estimate"] - np.linalg.norm(r)) <= rounding, params
        return s

    for its in (1, 5, 15, 16, 17, 32, 33):
        s = solve(ILS_RTOL=1e-15, ILS_MAX_NUM_ITERATIONS=its)
        assert not s.did_converge() and s.get_num_iterations() == its
    its = solve(ILS_RTOL=1e-9).get_num_iterations()   # and a limit that is just enough
    s = solve(ILS_RTOL=1e-9, ILS_MAX_NUM_ITERATIONS=its)
    assert s.did_converge() and s.get_num_iterations() == its
