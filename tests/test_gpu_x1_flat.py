"""The FP64 x1 sweep's blocks of 64 columns, which a launch of many columns of few
levels takes, against the oracle's fluxes, bit for bit: fewest levels and most,
columns that leave a remainder in the last block, scalars, both Riemann solvers,
and every number of waves a block may have."""
import numpy as np
import pytest

from helpers import atm_config, sw_config

pytestmark = pytest.mark.gpu


# 6 nx nx columns: at least 65,536, four blocks of 64 on each of 256 CUs
@pytest.mark.parametrize("nx, nx1, solver, ntracer", [
    (106, 3, 3, 0), (110, 4, 2, 1), (106, 24, 3, 0), (106, 25, 3, 0), (104, 3, 3, 0),
])
def test_x1_fluxes_are_the_oracles(ex, orc, nx, nx1, solver, ntracer):
    cfg = atm_config(ex, nx=nx, nx1=nx1, rsolver=solver, ntracer=ntracer)
    u0, s0 = ex.init_state(cfg, 1, nx + nx1)
    g, o = ex.Solver(cfg), orc.Oracle(cfg)
    for m in (g, o):
        m.upload(u0, s0)
        m.calc_fluxes()
    s, f = slice(3, 3 + nx), slice(3, 4 + nx1)
    want = o.flux(0)[:, :, s, s, f]
    assert np.array_equal(g.flux(0)[:, :, s, s, f], want)
    if ntracer:  # the scalars' fluxes are read through the state they make
        assert g.step(1) == o.step(1)
        assert np.array_equal(g.download()[1][:, :, s, s, 3:3 + nx1],
                              o.download()[1][:, :, s, s, 3:3 + nx1])
    g.close()
    o.close()


@pytest.mark.parametrize("waves", [2, 8])
def test_other_block_shapes(ex, waves):
    cfg = atm_config(ex, nx=106, nx1=5, implicit=0)
    u0, _ = ex.init_state(cfg, 1, 8)
    g, twin = ex.Solver(cfg), ex.Solver(cfg)
    for m in (g, twin):
        m.upload(u0)
    b = ex.Batch([g])
    b.set_caps({"x1_shape": waves, "x1": 300})
    b.step(2)
    twin.step(2)
    assert np.array_equal(g.download()[0], twin.download()[0])
    b.close()
    g.close()
    twin.close()


def test_beside_far_taller_members(ex):
    """the sweep's LDS is its own members': a batch with a tall mixed atmosphere
    and many layers of water, each of which would ask for more than a CU has"""
    mixed = atm_config(ex, nx=4, nx1=120)
    mixed.precision = ex.PREC_MIXED
    cfgs = [(atm_config(ex, nx=106, nx1=3), 1), (mixed, 1), (sw_config(ex, nx=4, nx1=300), 0)]
    members, twins = [], []
    for cfg, kind in cfgs:
        u0, _ = ex.init_state(cfg, kind, 4)
        for to in (members, twins):
            m = ex.Solver(cfg)
            m.upload(u0)
            to.append(m)
    b = ex.Batch(members)
    b.step(2, 0.5)
    for m, twin in zip(members, twins):
        twin.step(2, 0.5)
        assert np.array_equal(m.download()[0], twin.download()[0])
    b.close()
    for m in members + twins:
        m.close()
