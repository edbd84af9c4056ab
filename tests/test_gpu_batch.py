"""Batched form: every problem of a mixed batch assembled in one launch and
solved in one persistent launch, checked against the oracle per problem.

Gates: CSR pattern bit-exact and values/RHS within 1e-12 relative of the
oracle's assembly of the same mesh (2-D/3-D Q1, constant k, manufactured
source); FP64 true residual <= rtol ||b|| (checked on the host with the
oracle's matrix); solution within 1e-5 relative of the oracle's FP64 CG
solution to 1e-12 (the FP32-refined solve stops at rtol = 1e-8)."""
import numpy as np
import pytest

import fempar_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu

PROBLEMS = [(2, 4, 1.0, 1.0), (2, 7, 0.1, 1.0), (3, 3, 2.5, 1.0), (2, 16, 9.0, 1.0), (3, 5, 0.7, 2.0),
            (2, 33, 3.3, 1.0), (3, 8, 1.2, 1.0), (2, 2, 1.0, 1.0), (3, 11, 4.0, 0.5), (2, 64, 0.5, 1.0),
            (3, 16, 7.5, 1.0), (2, 100, 1.0, 1.0), (3, 2, 3.0, 1.0)]   # n = 2: one row, aliased offsets


def _oracle(dim, n, k, f0):
    sp = O.Space(O.make_problem(dim, [n] * dim, 1))
    ph = O.make_physics(k_kind=O.K_CONST, k0=k, f_kind=O.F_CELL_SIN, f0=f0)
    return sp.assemble(ph, symmetric_storage=False)


@pytest.fixture(scope="module")
def batch(env):
    b = F.batch_t(env, PROBLEMS, rtol=1e-8)
    b.assemble()
    yield b
    b.free()


def test_batch_matrices_match_oracle(batch):
    for i, (dim, n, k, f0) in enumerate(PROBLEMS):
        irp, ja, val, rhs = _oracle(dim, n, k, f0)
        birp, bja, bval, brhs = batch.get_problem_matrix(i)
        assert np.array_equal(birp, irp) and np.array_equal(bja, ja), (dim, n)
        if len(val):
            assert np.max(np.abs(bval - val)) <= 1e-12 * np.max(np.abs(val)), (dim, n)
            assert np.max(np.abs(brhs - rhs)) <= 1e-12 * np.max(np.abs(rhs)), (dim, n)


def test_batch_solutions(batch):
    for rep in range(2):        # the hipGraph is replayed: same answers
        print(f"[batch] solve replay {rep} of {len(PROBLEMS)} problems", flush=True)
        res = batch.solve()
        print(f"[batch] replay {rep}: {res['ms']:.3f} ms, iterations {res['num_iterations'].tolist()}", flush=True)
        assert np.all(res["did_converge"] == 1)
        assert np.all(res["latency_us"] > 0) and res["ms"] > 0
        for i, (dim, n, k, f0) in enumerate(PROBLEMS):
            irp, ja, val, rhs = _oracle(dim, n, k, f0)
            x = batch.get_solution(i)
            r = rhs - O.spmv(irp, ja, val, x, False)
            assert np.linalg.norm(r) <= 1.0001e-8 * np.linalg.norm(rhs), (dim, n)
            assert abs(res["true_residual"][i] - np.linalg.norm(r)) <= 1e-6 * np.linalg.norm(rhs) + 1e-300
            x_ref, info = O.cg(irp, ja, val, rhs, False, precond="jacobi", rtol=1e-12, maxit=20000)
            assert np.linalg.norm(x - x_ref) <= 1e-5 * np.linalg.norm(x_ref), (dim, n)
        if rep == 0:
            first = [batch.get_solution(i) for i in range(len(PROBLEMS))]
        else:
            for i in range(len(PROBLEMS)):
                assert np.array_equal(first[i], batch.get_solution(i))


def test_batch_autotune(batch):
    print("[batch] autotune", flush=True)
    t = batch.autotune()
    assert t in (256, 512, 1024)
    res = batch.solve()
    assert np.all(res["did_converge"] == 1)


# the sizes on both sides of each step between the ways a problem is solved
# (one wave, one workgroup of 256 or 1024 threads, passes over all problems),
# one batch for the small ones alone and one for the passes alone
@pytest.mark.parametrize("problems", [
    [(2, n, 0.3 + 0.1 * n, 1.0) for n in (3, 22, 23, 43, 44, 129, 130, 257)] +
    [(3, n, 5.0 - 0.1 * n, 2.0) for n in (4, 9, 10, 12, 13, 23, 24, 33)],
    [(2, 5, 1.0, 1.0), (3, 5, 2.0, 1.0)],
    [(3, 25, 2.0, 1.0), (2, 140, 0.5, 1.0)]], ids=["edges", "small", "passes"])
def test_batch_paths_match_oracle(env, problems):
    b = F.batch_t(env, problems, rtol=1e-8)
    b.assemble()
    res = b.solve()
    assert np.all(res["did_converge"] == 1) and np.all(res["latency_us"] > 0)
    for i, (dim, n, k, f0) in enumerate(problems):
        irp, ja, val, rhs = _oracle(dim, n, k, f0)
        x = b.get_solution(i)
        r = rhs - O.spmv(irp, ja, val, x, False)
        assert np.linalg.norm(r) <= 1.0001e-8 * np.linalg.norm(rhs), (dim, n)
        assert abs(res["true_residual"][i] - np.linalg.norm(r)) <= 1e-6 * np.linalg.norm(rhs), (dim, n)
        x_ref, _ = O.cg(irp, ja, val, rhs, False, precond="jacobi", rtol=1e-12, maxit=20000)
        assert np.linalg.norm(x - x_ref) <= 1e-5 * np.linalg.norm(x_ref), (dim, n)
    b.free()


def test_batch_problem_beyond_one_window(env):
    """A cube of 513^3 rows (1.08 GB a vector, more than 30-bit byte offsets reach)
    beside a small problem.  The source is the operator's lowest eigenvector, so the
    solution is known in closed form and its relative error is at most the
    relative residual, 1e-8 (and 1e-12 of rounding)."""
    n = 514
    print(f"[batch] one problem of {(n - 1) ** 3} rows", flush=True)
    b = F.batch_t(env, [(3, n, 2.0, 0.5), (2, 40, 1.0, 1.0)], rtol=1e-8)
    b.assemble()
    res = b.solve()
    print(f"[batch] solved in {res['ms']:.2f} ms, {res['num_iterations'].tolist()}", flush=True)
    assert np.all(res["did_converge"] == 1)
    for i, (dim, n, f0) in enumerate(((3, n, 0.5), (2, 40, 1.0))):
        h, g = 1.0 / n, 0.5 - 0.5 / np.sqrt(3.0)
        c = np.cos(np.pi * h)
        stiff, mass = 2.0 * (1.0 - c) / h, h * (2.0 + c) / 3.0        # of sin(pi x) at a node, by its value there
        load = h * ((1.0 - g) * np.cos(np.pi * h * g) + g * np.cos(np.pi * h * (1.0 - g)))
        scale = f0 * dim * np.pi ** 2 * load ** dim / (dim * stiff * mass ** (dim - 1))
        s = np.sin(np.pi * h * np.arange(1, n))
        ref = scale * s
        for _ in range(dim - 1):
            ref = np.multiply.outer(s, ref)
        x = b.get_solution(i).reshape(ref.shape)
        norm = np.linalg.norm(ref)
        x -= ref
        assert np.linalg.norm(x) <= (1e-8 + 1e-12) * norm, (dim, n)
        # no row is left out: the first and the last planes by themselves
        for plane in (0, n // 2, n - 2):
            assert np.linalg.norm(x[plane]) <= (1e-8 + 1e-12) * norm and np.linalg.norm(ref[plane]) > 0.0
    b.free()
