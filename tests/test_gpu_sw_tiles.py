"""Every kernel of the fused shallow-water stage on both sides of the number of
tiles (one a CU) from which a tile has 256 threads instead of 512: FP64 against
the oracle, mixed against the single phases, which take the same faces from
separate kernels, bit for bit; each Riemann solver alone and both in one batch."""
import numpy as np
import pytest

from helpers import interior, sw_config

pytestmark = pytest.mark.gpu
CUS = 256  # of the MI355X


def tiles(cfg):
    return 6 * cfg.nx1 * -(-cfg.nx // 16) * -(-cfg.nx // 15)


def water(ex, nx, nx1, solver, mixed):
    cfg = sw_config(ex, nx=nx, nx1=nx1, rsolver=solver)
    cfg.precision = ex.PREC_MIXED if mixed else ex.PREC_FP64
    return cfg


def loaded(ex, cfg):
    u0, _ = ex.init_state(cfg, 0, 31 * cfg.nx + cfg.rsolver)
    g = ex.Solver(cfg)
    g.upload(u0)
    return g, u0


def by_phases(ex, orc, cfg, dt):
    g, u0 = loaded(ex, cfg)
    if cfg.precision == ex.PREC_FP64:
        o = orc.Oracle(cfg)
        o.upload(u0)
        o.step(2, dt)
        u = o.download()[0]
        o.close()
    else:
        for _ in range(2):
            for stage in (1, 2, 3):
                g.stage(stage, dt)
        u = g.download()[0]
    g.close()
    return interior(u, cfg.nx1)


@pytest.mark.parametrize("nx, nx1, many", [(8, 1, False), (64, 3, True), (98, 1, True)])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("solver", [0, 1])
def test_stage_kernels(ex, orc, nx, nx1, many, mixed, solver):
    cfg = water(ex, nx, nx1, solver, mixed)
    assert (tiles(cfg) > CUS) == many
    g, _ = loaded(ex, cfg)
    g.step(2, 10.0)
    assert np.array_equal(interior(g.download()[0], nx1), by_phases(ex, orc, cfg, 10.0))
    g.close()


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("sizes", [((8, 1), (12, 1)), ((64, 3), (98, 1))])
def test_both_solvers_in_one_batch(ex, orc, sizes, mixed):
    cfgs = [water(ex, nx, nx1, q, mixed) for q, (nx, nx1) in enumerate(sizes)]
    members = [loaded(ex, c)[0] for c in cfgs]
    b = ex.Batch(members)
    b.step(2, 10.0)
    for m, c in zip(members, cfgs):
        assert np.array_equal(interior(m.download()[0], c.nx1), by_phases(ex, orc, c, 10.0))
    b.close()
    for m in members:
        m.close()
