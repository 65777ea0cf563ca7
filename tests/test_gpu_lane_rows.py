"""The batched engine's step over lane rows: a team too small for its registers
(64 threads, more than one or two reduction blocks) takes the general step
instead, whose results must be the same to the bit.  Sizes at the edges of
reduction blocks, row slices and the LDS layout (MPC: n = 16 N + 12), and
problems with long rows of A."""
import numpy as np
import pytest

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
