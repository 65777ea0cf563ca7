"""The batched engine's step over lane rows: a team too small for its registers
(64 threads, more than one or two reduction blocks) takes the general step
instead, whose results must be the same to the bit.  Sizes at the edges of
reduction blocks, row slices and the LDS layout (MPC: n = 16 N + 12), and
problems with long rows of A."""
import numpy as np
import pytest
import scipy.sparse as sp

from osqp_amd import problems as pr

pytestmark = pytest.mark.gpu

CASES = [("mpc", 1), ("mpc", 15), ("mpc", 16), ("mpc", 32), ("mpc", 63), ("mpc", 64), ("mpc", 90),
         ("portfolio", 100), ("portfolio", 511), ("portfolio", 1000)]


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("kind,size", CASES)
def test_teams_agree(kind, size, precision):
    from osqp_amd.serve import BatchEngine
    p = pr.mpc(size, seed=size) if kind == "mpc" else pr.portfolio(size, seed=size)
    out = []
    for team in (64, 256, 512):
        eng = BatchEngine(precision=precision, arena_bytes=1 << 28, eps_abs=1e-4, eps_rel=1e-4, max_iter=300)
        for b in range(3):
            eng.set_team(b, team, 2)
        r = eng.solve_batch([p])[0]
        out.append((r.x, r.y, r.info.iter, r.info.cg_iters, r.info.status_val, r.info.obj_val))
        eng.close()
    for o in out[1:]:
        assert o[2:] == out[0][2:]
        np.testing.assert_array_equal(o[0], out[0][0])
        np.testing.assert_array_equal(o[1], out[0][1])
    assert np.isfinite(out[0][0]).all()


def _with_empty_row(p):
    """The same QP with a free empty row last, which keeps it off lane rows."""
    A = sp.vstack([p["A"], sp.csc_matrix((1, p["A"].shape[1]))], format="csc")
    return dict(p, A=A, l=np.append(p["l"], -np.inf), u=np.append(p["u"], np.inf))


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("kind,size", CASES)
def test_row_groups_agree(kind, size, precision):
    """The lane rows' kernel and the row groups' on one problem: the same bits (long rows of A among them)."""
    from osqp_amd.serve import BatchEngine
    p = pr.mpc(size, seed=size) if kind == "mpc" else pr.portfolio(size, seed=size)
    m, out = p["A"].shape[0], []
    for q in (p, _with_empty_row(p)):
        eng = BatchEngine(precision=precision, arena_bytes=1 << 28, eps_abs=1e-4, eps_rel=1e-4, max_iter=300)
        r = eng.solve_batch([q])[0]
        # (a portfolio of 100 assets has medium rows: on row groups either way)
        assert eng.lanes() == (1, int(q is p and (kind, size) != ("portfolio", 100)))
        out.append((r.x, r.y[:m], r.info.iter, r.info.cg_iters, r.info.status_val, r.info.obj_val))
        eng.close()
    assert out[0][2:] == out[1][2:]
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])


def _resident(probs, precision, arena):
    """Adds resident problems and steps until nothing moves; the results of those that ended, in order."""
    from osqp_amd.serve import BatchEngine
    eng = BatchEngine(precision=precision, arena_bytes=arena, eps_abs=1e-4, eps_rel=1e-4, max_iter=300)
    ids = eng.add_many(probs, resident=True)
    done = {}
    for _ in range(400):
        ended = eng.step()
        for i in ended:
            done[i] = eng.poll(i)
        if not ended and eng.pending() == len(probs) - len(done) and len(done) == eng.lanes()[0]:
            break
    lanes = eng.lanes()
    eng.close()
    return [done.get(i) for i in ids], lanes


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("kind", ["mpc", "band"])
def test_an_arena_holds_as_many_problems(kind, precision):
    """An arena holds at least as many resident problems with lane rows as it does of the same without; where
    the lane rows' own arena is full, they run on row groups, and the results are those of a roomy engine."""
    rng = np.random.default_rng(1)
    if kind == "mpc":
        probs = [pr.mpc(30, seed=s) for s in range(24)]
    else:  # rows of three entries: the lane rows' copies are larger than the rest
        n = 500
        probs = [dict(P=sp.diags(1.0 + rng.random(n), format="csc"), q=rng.standard_normal(n),
                      A=sp.csc_matrix(sp.diags([rng.random(n), rng.random(n - 1), rng.random(n - 2)], [0, 1, 2])),
                      l=-rng.random(n), u=rng.random(n)) for _ in range(24)]
    arena = 8 << 20 if kind == "mpc" else 3 << 20
    roomy, on = _resident(probs, precision, 1 << 28)
    groups, off = _resident([_with_empty_row(p) for p in probs], precision, arena)
    tight, mixed = _resident(probs, precision, arena)
    assert on == (24, 24) and off[1] == 0 and 0 < off[0] < 24
    # (the lane arena, as large as the other, runs out first for the bands' FP32 copies alone)
    assert mixed[0] >= off[0] and mixed[1] > 0 and (mixed[1] < mixed[0]) == (kind == "band" and precision == 32)
    assert sum(r is not None for r in tight) == mixed[0]
    for a, b in zip(roomy, tight):
        if b is not None:
            assert a.info.iter == b.info.iter and a.info.status_val == b.info.status_val == 1
            np.testing.assert_array_equal(a.x, b.x)
            np.testing.assert_array_equal(a.y, b.y)


def test_a_problem_that_fits_on_row_groups_is_accepted():
    """An arena of a problem's size on row groups takes it, resident or not."""
    from osqp_amd.serve import BatchEngine
    p = pr.mpc(50, seed=3)  # 0.95 MiB
    for resident in (False, True):
        eng = BatchEngine(precision=32, arena_bytes=1 << 20, max_active=4, eps_abs=1e-4, eps_rel=1e-4)
        i = eng.add(p["P"], p["q"], p["A"], p["l"], p["u"], resident=resident)
        while eng.pending():
            eng.step()
        assert eng.poll(i).info.status_val == 1
        eng.close()
