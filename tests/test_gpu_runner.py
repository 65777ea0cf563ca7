"""The ADMM runner (many iterations in one launch, osqp_amd/csrc/hip/runner.h)
against the separate kernels, which a solver with section markers
(profiler_level 1) runs.

One workgroup: the runner takes every row and dot product in the separate
kernels' order, so x, y and the counts are the same bits.  Several workgroups:
other summation orders, and A x64 in FP64 recomputed in one iteration of eight.
FP64: 60 fixed iterations, whose linear solves take the same number of CG
iterations; the iterates then differ by accumulated rounding, at most 1e-9 as
observed (no bound is derived: K spans sigma 1e-6 to rho 1e2).  FP32: both
points meet their termination test, checked by their FP64 KKT certificates.
Each case asserts how many iterations the runner took, by how many workgroups.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from osqp_amd import OSQP
from osqp_amd import problems as pr

pytestmark = pytest.mark.gpu

EPS = dict(eps_abs=1e-4, eps_rel=1e-4)


def qp(n, m, row, seed, p_row=3, long_rows=0):
    """Random QP with about `row` entries a row of A; the first `long_rows` rows full."""
    rng = np.random.default_rng(seed)
    M = sp.random(n, n, density=min(1.0, p_row / n), random_state=rng, data_rvs=rng.standard_normal, format="csc")
    A = sp.random(m, n, density=min(1.0, row / n), random_state=rng, data_rvs=rng.standard_normal, format="lil")
    for r in range(long_rows):
        A[r, :] = rng.standard_normal(n)
    return dict(P=sp.triu(M @ M.T + 1e-2 * sp.eye(n), format="csc"), q=rng.standard_normal(n), A=sp.csc_matrix(A),
                l=-rng.random(m), u=rng.random(m), q2=rng.standard_normal(n))


def both(p, precision, second=None, **st):
    """(x, y, iter, status) of a solve and of a changed re-solve, the CG iterations and the run_stats, by the
    separate kernels and by the runner."""
    out = []
    for level in (1, 0):
        s = OSQP(precision=precision)
        assert s.setup(p["P"], p["q"], p["A"], p["l"], p["u"], profiler_level=level, **st) == 0
        res = []
        for change in (None, second):
            if change:
                s.update(**change)
            r = s.solve()
            res.append((r.x, r.y, r.info.iter, r.info.status_val))
        res += [s.stats().pcg_iters, s.run_stats()]
        s.close()
        out.append(res)
    assert (out[0][3].groups, out[0][3].iters) == (0, 0)
    return out


def ran(r, groups):
    """All iterations but each solve's first ran in launches of that many workgroups (0: none did)."""
    iters = sum(s[2] - 1 for s in r[:2]) if groups else 0
    assert (r[3].groups, r[3].iters, r[3].failed) == (groups, iters, 0)


# (n, m, entries a row, full rows): lone elements, odd and RB-divisible n, the
# workgroup's width and one above, rows past a panel task, an empty row
ONE = [(1, 1, 1, 0), (2, 3, 1, 0), (63, 65, 3, 0), (255, 400, 4, 1), (256, 300, 4, 0), (500, 64, 5, 1), (801, 90, 6, 2),
       (1023, 700, 5, 0), (1024, 1025, 5, 0), (1025, 600, 6, 0), (2047, 300, 3, 0), (2048, 40, 8, 1)]
# one full row among short ones in a slice: padded past what the layout takes, on the separate kernels
PADDED = {(255, 400, 64), (255, 400, 32), (500, 64, 32)}


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n,m,row,full", ONE)
def test_one_workgroup_same_bits(n, m, row, full, precision):
    p = qp(n, m, row, seed=n + m, p_row=1.5, long_rows=full)
    new_A = np.random.default_rng(1).standard_normal(p["A"].nnz)
    a, b = both(p, precision, second=dict(q=p["q2"], Ax=new_A), **EPS)
    ran(b, 0 if (n, m, precision) in PADDED else 1)
    assert a[2] == b[2]
    for u, v in zip(a[:2], b[:2]):
        assert u[2:] == v[2:]
        assert np.array_equal(u[0], v[0]) and np.array_equal(u[1], v[1])


# past horizon 92 (n + m = 4084) [P A'] has two column panels, whose order the one workgroup does not keep
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("N", [10, 33, 50, 92, 93, 127])
def test_mpc_same_bits(N, precision):
    p = pr.mpc(N, seed=N)
    l, u = p["l"].copy(), p["u"].copy()
    l[:12] = u[:12] = np.random.default_rng(N).uniform(-1, 1, 12)
    a, b = both(p, precision, second=dict(l=l, u=u), **EPS)
    ran(b, 1 if N <= 92 else 0)
    assert a[2] == b[2]
    for s, t in zip(a[:2], b[:2]):
        assert s[2:] == t[2:] and np.array_equal(s[0], t[0]) and np.array_equal(s[1], t[1])


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n,m,row", [(64, 4032, 4), (64, 4033, 4), (40, 9000, 3)])
def test_tall_with_equality_rows_same_bits(n, m, row, precision):
    p = qp(n, m, row, seed=m)
    x = np.random.default_rng(3).uniform(-0.1, 0.1, n)
    p["l"][:5] = p["u"][:5] = (p["A"] @ x)[:5]
    a, b = both(p, precision, second=dict(q=p["q2"]), **EPS)
    ran(b, 1 if n + m <= 4096 else 0)
    assert a[2] == b[2]
    for s, t in zip(a[:2], b[:2]):
        assert s[2:] == t[2:] and np.array_equal(s[0], t[0]) and np.array_equal(s[1], t[1])


# (n, m, entries a row, workgroups): 32, 64, 128 and 256 workgroups; 1 to 12 elements a
# thread; fewer columns than workgroups; more rows than threads a workgroup
MANY = [(200, 4000, 20, 32), (33, 30000, 5, 64), (700, 9001, 30, 64), (1025, 12000, 40, 128), (2049, 9000, 90, 128),
        (4097, 30001, 70, 256), (6145, 20000, 30, 128), (8191, 24000, 25, 128)]


@pytest.mark.parametrize("n,m,row,groups", MANY)
def test_many_workgroups_fp64(n, m, row, groups):
    p = qp(n, m, row, seed=n)
    a, b = both(p, 64, second=dict(q=p["q2"]), eps_abs=1e-30, eps_rel=1e-30, max_iter=60)
    ran(b, groups)
    assert a[2] == b[2]
    for u, v in zip(a[:2], b[:2]):
        assert u[2:] == v[2:]
        for k in (0, 1):
            assert np.linalg.norm(u[k] - v[k]) <= 1e-9 * max(1.0, np.linalg.norm(u[k]))


@pytest.mark.parametrize("n,m,row,groups", MANY + [(9001, 30000, 25, 128), (12288, 40000, 20, 128)])
def test_many_workgroups_fp32(n, m, row, groups):
    p = qp(n, m, row, seed=n)
    a, b = both(p, 32, second=dict(l=p["l"] - 0.1, u=p["u"] + 0.1), **EPS)
    ran(b, groups)
    for k, prob in enumerate((p, dict(p, l=p["l"] - 0.1, u=p["u"] + 0.1))):
        assert a[k][3] == b[k][3] and a[k][3] in (1, 2, 7)
        if a[k][3] == 7:  # 33 x 30000 stops at max_iter, as the separate kernels do: no test to certify, the same point
            assert n == 33 and a[k][2] == b[k][2] == 4000
            for u, v in zip(a[k][:2], b[k][:2]):
                assert np.linalg.norm(u - v) <= 1e-3 * np.linalg.norm(u)
            continue
        eps = 1e-4 if a[k][3] == 1 else 1e-3  # solved inaccurate: ten times the tolerances
        for x, y, _, _ in (a[k], b[k]):
            c = pr.kkt_certificate(prob, x, y)
            assert c["prim"] <= eps + eps * c["scale_p"]
            assert c["dual"] <= eps + eps * c["scale_d"]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("check", [25, 0])
def test_a_wait_that_gives_up_is_done_again(precision, check):
    """Waits that give up at once (every workgroup leaves its launch): the iterations of that launch are
    done again by the separate kernels, so the solve and the next one are theirs to the bit."""
    p = qp(700, 9001, 30, seed=9)
    # without checks and rho updates the host sees nothing of a run but whether it gave up
    st = dict(EPS, check_termination=check, **({} if check else dict(adaptive_rho=0, max_iter=100)))
    out = []
    for polls in (None, 0):
        s = OSQP(precision=precision)
        assert s.setup(p["P"], p["q"], p["A"], p["l"], p["u"], profiler_level=1 if polls is None else 0, **st) == 0
        if polls is not None:
            assert s.run_stats().groups > 1
            s.run_polls(polls)
        r = []
        for q in (p["q"], p["q2"]):
            s.update(q=q)
            r.append(s.solve())
            assert r[-1].rc == 0
        out.append((r, s.stats().pcg_iters, s.run_stats()))
        s.close()
    (a, na, sa), (b, nb, sb) = out
    assert (sa.iters, sa.failed) == (0, 0) and (sb.iters, sb.failed, sb.groups) == (0, 1, 0)
    assert na == nb
    for u, v in zip(a, b):
        assert (u.info.iter, u.info.status_val) == (v.info.iter, v.info.status_val)
        assert np.array_equal(u.x, v.x) and np.array_equal(u.y, v.y)
        for f in ("prim_res", "dual_res", "obj_val", "primdual_int", "rho_updates"):
            assert getattr(u.info, f) == getattr(v.info, f)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n,m,row,long", [(400, 70000, 3, 60), (400, 70000, 3, 24), (2500, 9000, 12, 300)])
def test_no_lane_adds_up_a_long_row(n, m, row, long, precision):
    """Rows far longer than the average: their entries are spread over lanes, at most 24 a lane, as over the
    lanes of a panel task, and the iterates are the separate kernels'."""
    p = qp(n, m, row, seed=m)
    A = p["A"].tolil()
    for r in range(0, m, m // 40):
        A[r, :long] = np.random.default_rng(r).standard_normal(long)
    p["A"] = sp.csc_matrix(A)
    a, b = both(p, precision, second=dict(q=p["q2"]), eps_abs=1e-30, eps_rel=1e-30, max_iter=40)
    assert b[3].groups > 1 and b[3].iters == 78 and 1 <= b[3].chain <= 24
    for u, v in zip(a[:2], b[:2]):
        assert np.linalg.norm(u[0] - v[0]) <= (1e-9 if precision == 64 else 1e-3) * max(1.0, np.linalg.norm(u[0]))


def test_rows_out_of_order_stay_on_the_separate_kernels(monkeypatch):
    """Columns whose rows are not ascending, as a C caller may pass them: the several-workgroup layout needs
    the order, so the solve takes the separate kernels and gives the sorted problem's answer."""
    from osqp_amd import solver

    class Reversed(solver.T.CscHolder):
        def __init__(self, M):
            super().__init__(M.copy())
            if self.m != self.n:
                for j in range(self.n):
                    c = slice(self.p[j], self.p[j + 1])
                    self.i[c], self.x[c] = self.i[c][::-1].copy(), self.x[c][::-1].copy()

    p = qp(300, 5000, 12, seed=4)
    r = {}
    for name in ("sorted", "reversed"):
        if name == "reversed":
            monkeypatch.setattr(solver.T, "CscHolder", Reversed)
        s = OSQP(precision=64)
        assert s.setup(p["P"], p["q"], p["A"], p["l"], p["u"], **EPS) == 0
        assert s.run_stats().groups == (32 if name == "sorted" else 0)
        r[name] = s.solve()
        s.close()
    assert r["sorted"].info.status_val == r["reversed"].info.status_val == 1
    assert np.linalg.norm(r["sorted"].x - r["reversed"].x) <= 1e-3 * np.linalg.norm(r["sorted"].x)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("features", [500, 620])
def test_equality_rows_keep_the_separate_kernels_order(features, precision):
    """A lasso's equality rows (too many entries for one workgroup): the same bits as the separate kernels;
    relaxed to inequalities, the several-workgroup kernel's solve ends at a certified point."""
    p = pr.lasso(features, 10 * features + 3, 0.02, seed=features)
    relaxed = dict(l=p["l"] - 0.05, u=p["u"] + 0.05)
    a, b = both(p, precision, second=relaxed, **EPS)
    # the lasso's FP32 operators are no panels: both its solves keep the separate kernels
    assert (b[3].groups > 1, b[3].iters) == ((True, b[1][2] - 1) if precision == 64 else (False, 0))
    assert a[0][2:] == b[0][2:]
    assert np.array_equal(a[0][0], b[0][0]) and np.array_equal(a[0][1], b[0][1])
    assert a[1][3] == b[1][3] == 1
    c = pr.kkt_certificate(dict(p, **relaxed), b[1][0], b[1][1])
    assert c["prim"] <= 1e-4 + 1e-4 * c["scale_p"] and c["dual"] <= 1e-4 + 1e-4 * c["scale_d"]


@pytest.mark.parametrize("precision", [64, 32])
def test_built_where_it_can_run(precision):
    """With equality rows the several-workgroup kernel is not built; it is once they are gone, and a solver
    that never iterates many at a time builds none."""
    p = qp(700, 9001, 30, seed=2)
    ax = p["A"] @ np.random.default_rng(3).uniform(-0.01, 0.01, 700)
    l, u = p["l"].copy(), p["u"].copy()
    l[:5] = u[:5] = ax[:5]
    s = OSQP(precision=precision)
    assert s.setup(p["P"], p["q"], p["A"], l, u, **EPS) == 0
    assert s.run_stats().groups == 0
    s.solve()
    assert (s.run_stats().groups, s.run_stats().iters) == (0, 0)
    s.update(l=p["l"], u=p["u"])
    r = s.solve()
    assert s.run_stats().groups > 1 and s.run_stats().iters == r.info.iter - 1
    s.update(l=l, u=u)  # equality rows again: built, not used
    s.solve()
    assert s.run_stats().iters == r.info.iter - 1
    s.close()
    q = qp(300, 3000, 20, seed=2)
    for st, groups in ((dict(), True), (dict(time_limit=100.0), False), (dict(profiler_level=1), False)):
        s = OSQP(precision=precision)
        assert s.setup(q["P"], q["q"], q["A"], q["l"], q["u"], **EPS, **st) == 0
        s.solve()
        assert (s.run_stats().groups > 1, s.run_stats().iters > 0) == (groups, groups)
        s.close()
