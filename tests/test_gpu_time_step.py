"""The CFL time step's block-wise minimum against the oracle, called again and
again on one handle (each call leaves the words of the minimum as the next finds
them): one block, the 32 lines the blocks are counted over less one, all, and one
more, and several blocks a line."""
import numpy as np
import pytest

from helpers import atm_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx, nx1", [(4, 3), (34, 9), (60, 3), (22, 23), (64, 12)])
def test_repeated_time_steps_are_the_oracles(ex, orc, nx, nx1):
    cfg = atm_config(ex, nx=nx, nx1=nx1)
    cfg.cfl_x1 = 0
    u0, _ = ex.init_state(cfg, 1, nx)
    g, o = ex.Solver(cfg), orc.Oracle(cfg)
    rng = np.random.default_rng(nx)
    for _ in range(4):
        u = u0.copy()  # one hot cell, the minimum's, somewhere else each time
        at = rng.integers(6), 3 + rng.integers(nx), 3 + rng.integers(nx), 3 + rng.integers(nx1)
        u[at[0], 4, at[1], at[2], at[3]] *= 4
        for m in (g, o):
            m.upload(u)
        want = o.new_dt()
        assert [g.new_dt() for _ in range(12)] == [want] * 12
    g.close()
    o.close()
