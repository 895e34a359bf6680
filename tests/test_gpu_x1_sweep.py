"""The FP64 x1 sweep (blocks of 16 columns, or of 8 on a launch of few) against
the oracle's fluxes, bit for bit: panels whose columns leave a remainder in the
last block, the fewest levels and more than a block works on at once, passive
scalars, both Riemann solvers, with and without the hydrostatic decomposition."""
import numpy as np
import pytest

from helpers import atm_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx, nx1, solver, ntracer, grav", [
    (4, 3, 3, 0, -9.81), (6, 7, 2, 1, -9.81), (10, 70, 3, 2, -9.81), (6, 33, 3, 0, 0.0),
    (52, 4, 3, 0, -9.81), (54, 5, 2, 1, -9.81), (66, 3, 3, 0, 0.0),
])
def test_x1_fluxes_are_the_oracles(ex, orc, nx, nx1, solver, ntracer, grav):
    cfg = atm_config(ex, nx=nx, nx1=nx1, rsolver=solver, ntracer=ntracer)
    cfg.grav = grav
    u0, s0 = ex.init_state(cfg, 1, 31 * nx + nx1)
    g, o = ex.Solver(cfg), orc.Oracle(cfg)
    for m in (g, o):
        m.upload(u0, s0)
        m.fill_ghosts()
        m.calc_fluxes()
    s, f = slice(3, 3 + nx), slice(3, 4 + nx1)
    assert np.array_equal(g.flux(0)[:, :, s, s, f], o.flux(0)[:, :, s, s, f])
    if ntracer:  # the scalars' fluxes are read through the state they make
        assert g.step(1) == o.step(1)
        assert np.array_equal(g.download()[1][:, :, s, s, 3:3 + nx1],
                              o.download()[1][:, :, s, s, 3:3 + nx1])
    g.close()
    o.close()
