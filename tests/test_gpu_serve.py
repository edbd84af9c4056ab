"""Serving form: elasticity requests through the continuous-batching server.

Gates: each solution within 1e-6 relative of the oracle's FP64 CG solution
(to 1e-12) and its FP64 true residual <= rtol ||b|| on the oracle's matrix
(vector Q1, clamped on x = 0, body force (0, 0, -1); the oracle restates
sbm_irreducible_discrete_integration.i90:64-130 and cg.f90:101-407); every
result bit-identical alone and in a mix of requests in flight together;
admission never exceeds the HBM budget and refuses a request larger than it."""
import numpy as np
import pytest

import fempar_amd as F
from fempar_amd import _native as N
from oracle import oracle as O

pytestmark = pytest.mark.gpu

RTOL = 1e-8


def _oracle(n, E, nu):
    sp = O.Space(O.make_problem(3, (n, n, n), 1, 3, O.BC_X0))
    ph = O.make_physics(kind=O.PHYS_ELASTICITY, E=E, nu=nu, body=(0, 0, -1))
    return sp, sp.assemble(ph, False)


def _to_reference(sp, n, x_served):
    """The served solution (entry 3 v + c = component c of free vertex v, x index
    1..n fastest) in the oracle's first-touch numbering."""
    d = sp.dofs()                                   # cells x 24, local index c * 8 + vertex
    x = np.empty(sp.n_free)
    for cell in range(sp.num_cells):
        i, j, k = cell % n, (cell // n) % n, cell // (n * n)
        for l in range(24):
            g = d[cell, l]
            if g <= 0:
                continue
            c, vl = divmod(l, 8)
            a, b, z = i + (vl & 1), j + ((vl >> 1) & 1), k + (vl >> 2)
            v = (a - 1) + n * (b + (n + 1) * z)
            x[g - 1] = x_served[3 * v + c]
    return x


def test_serve_matches_oracle(env):
    srv = F.serve_t(env, max_active=4, setup_threads=2, rtol=RTOL)
    try:
        cases = [(2, 1.0, 0.3), (3, 50.0, 0.2), (4, 120.0, 0.45), (5, 7.5, 0.33)]
        tickets = [srv.submit(n, E, nu) for n, E, nu in cases]
        for t, (n, E, nu) in zip(tickets, cases):
            print(f"[serve] waiting for n={n} E={E} nu={nu}", flush=True)
            res = srv.wait(t, timeout_s=60)
            assert res["status"] == N.OK and res["did_converge"] == 1, res
            sp, (irp, ja, val, rhs) = _oracle(n, E, nu)
            assert res["num_dofs"] == len(rhs) == 3 * n * (n + 1) ** 2
            x = _to_reference(sp, n, srv.get_solution(t))
            r = rhs - O.spmv(irp, ja, val, x, False)
            assert np.linalg.norm(r) <= 1.0001 * RTOL * np.linalg.norm(rhs), (n, np.linalg.norm(r))
            # the reported FP64 residual is that of the returned solution (the two
            # sums differ only in rounding, far below the residual itself)
            assert res["true_residual"] > 0
            assert abs(res["true_residual"] - np.linalg.norm(r)) <= 1e-3 * np.linalg.norm(r) + 1e-13 * np.linalg.norm(rhs)
            assert abs(res["rhs_norm"] - np.linalg.norm(rhs)) <= 1e-12 * np.linalg.norm(rhs)
            x_ref, info = O.cg(irp, ja, val, rhs, False, precond="jacobi", rtol=1e-12, maxit=50000)
            assert info["converged"]
            assert np.linalg.norm(x - x_ref) <= 1e-6 * np.linalg.norm(x_ref), n
            assert 0 < res["hbm_bytes"] <= res["hbm_estimate"]
            assert res["latency_ms"] >= res["solve_ms"] > 0
            srv.release(t)
    finally:
        srv.free()


def test_serve_alone_vs_mixed(env):
    cases = [(3, 10.0, 0.25), (12, 80.0, 0.3), (6, 2.0, 0.4), (16, 150.0, 0.22), (4, 33.0, 0.44),
             (9, 1.5, 0.35), (14, 60.0, 0.28), (5, 190.0, 0.21)]
    srv = F.serve_t(env, max_active=8, setup_threads=4, rtol=RTOL)
    try:
        alone = []
        for n, E, nu in cases:
            t = srv.submit(n, E, nu)
            res = srv.wait(t, timeout_s=60)
            assert res["did_converge"] == 1, (n, res)
            alone.append((res, srv.get_solution(t)))
            srv.release(t)
        print("[serve] alone done; submitting the mix", flush=True)
        tickets = [srv.submit(n, E, nu) for n, E, nu in cases]
        for t, (n, E, nu), (ra, xa) in zip(tickets, cases, alone):
            res = srv.wait(t, timeout_s=120)
            assert res["status"] == N.OK, (n, res["status"], res["error"])
            x = srv.get_solution(t)
            assert res["num_iterations"] == ra["num_iterations"], n
            assert np.array_equal(x, xa), n          # same bits alone and in the mix
            srv.release(t)
        st = srv.stats()
        print(f"[serve] stats {st}", flush=True)
        assert st["completed"] == 2 * len(cases) and st["failed"] == 0
        assert st["running_peak"] >= 2              # requests iterated together
        # every request's buffers came from its block of the arena reserved at
        # creation: no device allocation while requests iterated
        assert st["arena_bytes"] > 0 and st["arena_fallbacks"] == 0
    finally:
        srv.free()


def test_serve_admission_budget(env):
    probe = F.serve_t(env, max_active=1, setup_threads=1)
    est4, est16 = probe.estimate_bytes(4), probe.estimate_bytes(16)
    probe.free()
    budget = 1.2 * est4                              # room for one n = 4 request at a time
    srv = F.serve_t(env, hbm_budget_bytes=budget, max_active=4, setup_threads=2, rtol=RTOL)
    try:
        with pytest.raises(N.FemhipError) as ei:
            srv.submit(16, 10.0, 0.3)
        assert ei.value.code == N.ERR_ADMISSION and est16 > budget
        tickets = [srv.submit(4, 10.0 + i, 0.3) for i in range(3)]
        for t in tickets:
            assert srv.wait(t, timeout_s=60)["did_converge"] == 1
            srv.release(t)
        st = srv.stats()
        assert st["peak_active"] == 1 and st["hbm_peak"] <= budget
        assert st["hbm_in_use"] == 0 and st["active"] == 0
        assert st["arena_bytes"] >= budget and st["arena_fallbacks"] == 0
    finally:
        srv.free()


def test_serve_errors(env):
    srv = F.serve_t(env, max_active=2, setup_threads=1)
    try:
        # n = 207 would overflow the operator's 32-bit entry index: refused at
        # submit, before it takes a slot or budget
        for bad in [dict(n=0, E=1.0, nu=0.3), dict(n=4, E=-1.0, nu=0.3), dict(n=4, E=1.0, nu=0.5),
                    dict(n=207, E=1.0, nu=0.3)]:
            with pytest.raises(N.FemhipError) as ei:
                srv.submit(**bad)
            assert ei.value.code == N.ERR_INVALID
        with pytest.raises(N.FemhipError):
            srv.wait(12345, timeout_s=0.1)
        # a future arrival is not admitted before its time
        t = srv.submit(2, 1.0, 0.3, arrival_s=srv.now() + 0.5)
        with pytest.raises(N.FemhipError) as ei:
            srv.wait(t, timeout_s=0.1)
        assert ei.value.code == N.ERR_STATE
        res = srv.wait(t, timeout_s=30)
        assert res["did_converge"] == 1 and res["queue_ms"] < 100.0
    finally:
        srv.free()


@pytest.mark.parametrize("policy,aging_s", [("fcfs", 0.0), ("smallest", 0.0), ("smallest", 1e-9)])
def test_serve_admission_order(env, policy, aging_s):
    """One slot, a large request submitted before three small ones, all arriving
    at the same instant: first come, first served admits the large one first;
    smallest-first admits the small ones first; with an aging bound already
    passed, arrival order wins again."""
    srv = F.serve_t(env, max_active=1, setup_threads=1, rtol=RTOL, admission=policy, aging_s=aging_s)
    try:
        t0 = srv.now() + 0.3
        big = srv.submit(16, 40.0, 0.3, arrival_s=t0)
        small = [srv.submit(3, 10.0 + i, 0.3, arrival_s=t0) for i in range(3)]
        rb = srv.wait(big, timeout_s=120)
        rs = [srv.wait(t, timeout_s=120) for t in small]
        assert rb["did_converge"] == 1 and all(r["did_converge"] == 1 for r in rs)
        small_first = all(r["queue_ms"] < rb["queue_ms"] for r in rs)
        print(f"[serve] {policy} aging={aging_s}: big queued {rb['queue_ms']:.1f} ms, "
              f"small {[round(r['queue_ms'], 1) for r in rs]}", flush=True)
        assert small_first == (policy == "smallest" and aging_s == 0.0)
    finally:
        srv.free()


def test_serve_reused_memory_and_padded_components(env):
    """Sizes whose components do not fill whole slices, in both forms of an
    iteration (70: more than a million rows), in a device block that an earlier
    request has written: the rows between the components take no part."""
    srv = F.serve_t(env, hbm_budget_bytes=4 << 30, max_active=1, setup_threads=1, rtol=RTOL)
    try:
        for n in (68, 70, 41, 72, 70):
            print(f"[serve] padded components, n={n}", flush=True)
            t = srv.submit(n, 50.0, 0.3)
            res = srv.wait(t, timeout_s=60)
            assert res["status"] == N.OK and res["did_converge"] == 1, (n, res)
            assert res["true_residual"] <= 1.0001 * RTOL * res["rhs_norm"], n
            x = srv.get_solution(t)
            assert np.all(np.isfinite(x)) and np.linalg.norm(x) > 0
            srv.release(t)
    finally:
        srv.free()
