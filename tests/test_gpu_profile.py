"""The measuring calls beside a solve: femhip_solver_profile_spmv leaves the last
solve's history and solution as they are, femhip_solver_profile_cg is a solve of
its own to the end.  A system whose CG runs in one workgroup, one whose products
are formed from the cells, and one on its stored matrix."""
import numpy as np
import pytest

import fempar_amd as F

pytestmark = pytest.mark.gpu

SYSTEMS = {"small": ((30, 31), 1, "boundary"), "cells": ((30, 31, 29), 1, "boundary"), "cells_q2": ((9, 10, 11), 2, "x0"),
           "stored": ((30, 31, 29), 1, "moved")}


def _operator(env, name):
    n, order, bc = SYSTEMS[name]
    tria = F.serial_triangulation_t().create(env, {
        "STRUCT_HEX_MESH_GENERATOR_NUM_DIMS": len(n), "STRUCT_HEX_MESH_GENERATOR_NUM_CELLS_X_DIM": list(n),
        "STRUCT_HEX_MESH_GENERATOR_DOMAIN_LIMITS": [0, 1] * len(n)})
    fes = F.serial_fe_space_t().create(tria, order=order, dirichlet="boundary" if bc == "moved" else bc)
    if bc == "moved":   # vertices given by the caller, though where they were
        vc = np.ascontiguousarray(tria.get_uniform_vertex_coordinates())
        F._native.check(fes._lib.femhip_space_set_vertex_coords(fes.h, F._native.ptr(vc)))
    op = F.fe_affine_operator_t()
    op.create("CSR", [True], fes, F.poisson_discrete_integration_t(k="const", k0=1.5, f="const", f0=2.0))
    op.compute()
    return op


def _solver(env, op, **params):
    s = F.iterative_linear_solver_t().create(env)
    s.set_type_from_string("CG")
    s.set_parameters_from_pl(params)
    s.set_operators(op, F.jacobi_preconditioner_t(op))
    return s


@pytest.mark.parametrize("name", SYSTEMS)
def test_profile_spmv_keeps_the_solve(env, name):
    print(f"[profile] spmv {name}", flush=True)
    op = _operator(env, name)
    s = _solver(env, op, ILS_RTOL=1e-8)
    s.solve_resident()
    its, x, hist = s.get_num_iterations(), s.get_solution(), s.get_error_estimate_history_convergence_test()
    assert len(hist) == its > 1
    ms, nbytes = s.profile_spmv(3)
    assert ms > 0 and nbytes > 0
    assert np.array_equal(s.get_error_estimate_history_convergence_test(), hist)
    assert np.array_equal(s.get_solution(), x)
    ms, count, nbytes = s.profile_cg()
    assert ms > 0 and nbytes > 0 and count == its
    again = s.get_error_estimate_history_convergence_test()   # of the profiled solve: the same one
    assert len(again) == its and np.max(np.abs(again / hist - 1.0)) <= 1e-7
    assert np.linalg.norm(s.get_solution() - x) <= 1e-10 * np.linalg.norm(x)


@pytest.mark.parametrize("precision", ["FP64", "FP32_REFINED"])
@pytest.mark.parametrize("name", SYSTEMS)
def test_profile_cg_runs_to_the_limit(env, name, precision):
    """A limit that is a whole number of chunks: the passes that decide an
    iteration after it, and those of an update, are launched all the same."""
    print(f"[profile] cg {name} {precision}", flush=True)
    op = _operator(env, name)
    s = _solver(env, op, ILS_RTOL=1e-14, ILS_MAX_NUM_ITERATIONS=32, FEMHIP_PRECISION=precision)
    s.solve_resident()
    assert not s.did_converge() and s.get_num_iterations() == 32
    x = s.get_solution()
    ms, count, _ = s.profile_cg()
    assert ms > 0 and count == 32
    assert np.linalg.norm(s.get_solution() - x) <= 1e-10 * np.linalg.norm(x)
