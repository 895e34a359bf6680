"""The column solves within and outside a stage against the oracle, bit for bit:
level counts that leave remainders of the three (5x5) and six (3x3) levels a
piece of the backward sweep holds and of the two levels the 3x3 assembly takes
at once, panels whose columns leave a remainder in the last block of
64, and both sides of the number of blocks (two a CU) above which a block has one
wave instead of several."""
import numpy as np
import pytest

from helpers import atm_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("implicit", [9, 1])
@pytest.mark.parametrize("nx, nx1", [(4, 3), (4, 4), (6, 5), (8, 6), (10, 17), (4, 8), (6, 10), (72, 4), (74, 3),
                                     (74, 5)])
def test_column_solve_is_the_oracles(ex, orc, nx, nx1, implicit):
    cfg = atm_config(ex, nx=nx, nx1=nx1, implicit=implicit)
    u0, _ = ex.init_state(cfg, 1, 17 * nx + nx1)
    g, o = ex.Solver(cfg), orc.Oracle(cfg)
    for m in (g, o):
        m.upload(u0)
    assert g.step(2, 5.0) == o.step(2, 5.0)
    s, i = slice(3, 3 + nx), slice(3, 3 + nx1)
    assert np.array_equal(g.download()[0][:, :, s, s, i], o.download()[0][:, :, s, s, i])
    dt = 5.0
    for m in (g, o):
        m.fill_ghosts()
        m.calc_fluxes()
        m.add_flux_divergence(dt)
        m.implicit_correct(dt)
    assert np.array_equal(g.download()[0][:, :, s, s, i], o.download()[0][:, :, s, s, i])
    g.close()
    o.close()
