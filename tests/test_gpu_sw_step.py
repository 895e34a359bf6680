"""The whole step of shallow water without scalars (k_sw_stage, k_sw_halo, the
panel-edge states beside k_dt) against the oracle, bit for bit in FP64, on panels
below, on and past the edges of its 16 x 15 tiles, with few tiles (512 threads a
tile) and many (256), stepped one at a time and from a replayed graph, and as
members of a batch of both equations of state.  The mixed form is held to 1e-6
of each variable's maximum: three steps of FP32 face deltas (2^-24 = 6e-8 of a
flux's variation, which is itself a fraction of the flux)."""
import numpy as np
import pytest

from helpers import atm_config, sw_config

pytestmark = pytest.mark.gpu


def face_ghosts_and_inner(shape, nx1):
    """cells the step defines: interior and face-ghost columns, interior levels"""
    m = np.zeros(shape[2:], bool)
    m[3:-3, :, 3:3 + nx1] = True
    m[:, 3:-3, 3:3 + nx1] = True
    return m


def start(ex, cfg):
    u0, _ = ex.init_state(cfg, 0, 100 + cfg.nx)
    g = ex.Solver(cfg)
    g.upload(u0)
    return g, u0


@pytest.mark.parametrize("nx, nx1, solver, coriolis", [
    (4, 1, 0, 1), (14, 2, 1, 0), (16, 1, 0, 2), (18, 1, 1, 1), (30, 1, 0, 1), (32, 1, 1, 2),
    (34, 2, 0, 1), (64, 3, 0, 1),
])
def test_step_is_the_oracles(ex, orc, nx, nx1, solver, coriolis):
    cfg = sw_config(ex, nx=nx, nx1=nx1, rsolver=solver, coriolis=coriolis)
    g, u0 = start(ex, cfg)
    o = orc.Oracle(cfg)
    o.upload(u0)
    dts = [g.step(1), g.step(3), g.step(2, 50.0)]  # eager; replayed; replayed, given dt
    assert dts == [o.step(1), o.step(3), o.step(2, 50.0)]
    m = face_ghosts_and_inner(u0.shape, nx1)
    assert np.array_equal(g.download()[0][:, :, m], o.download()[0][:, :, m])
    assert np.array_equal(g.prim()[:, :, m], o.prim()[:, :, m])
    # a single phase after the step reads the state the step left
    g.calc_fluxes()
    o.calc_fluxes()
    s = slice(3, 3 + nx)
    assert np.array_equal(g.flux(1)[:, :, s, 3:4 + nx, 3:3 + nx1],
                          o.flux(1)[:, :, s, 3:4 + nx, 3:3 + nx1])
    g.close()
    o.close()


@pytest.mark.parametrize("graph", [False, True])
def test_members_of_a_mixed_batch(ex, orc, graph):
    cfgs = [sw_config(ex, nx=18, nx1=1), atm_config(ex, nx=6, nx1=6),
            sw_config(ex, nx=34, nx1=1, rsolver=1)]
    sw = [0, 2]
    started = [start(ex, c) if q in sw else None for q, c in enumerate(cfgs)]
    air = ex.Solver(cfgs[1])
    air.upload(ex.init_state(cfgs[1], 1, 5)[0])
    members = [air if s is None else s[0] for s in started]
    b = ex.Batch(members, graph=graph)
    b.step(2)
    b.step(2)
    for q in sw:
        o = orc.Oracle(cfgs[q])
        o.upload(started[q][1])
        o.step(4)
        m = face_ghosts_and_inner(started[q][1].shape, cfgs[q].nx1)
        assert np.array_equal(members[q].download()[0][:, :, m], o.download()[0][:, :, m])
        o.close()
    b.close()


@pytest.mark.parametrize("nx, solver", [(4, 0), (16, 1), (34, 0), (96, 1)])
def test_mixed_step(ex, orc, nx, solver):
    cfg = sw_config(ex, nx=nx, nx1=1, rsolver=solver)
    cfg.precision = ex.PREC_MIXED
    g, u0 = start(ex, cfg)
    ref = sw_config(ex, nx=nx, nx1=1, rsolver=solver)
    o = orc.Oracle(ref)
    o.upload(u0)
    assert abs(g.step(3) / o.step(3) - 1) < 1e-6
    m = face_ghosts_and_inner(u0.shape, 1)
    a, b = g.download()[0][:, :, m], o.download()[0][:, :, m]
    for n in (0, 2, 3):
        assert np.abs(a[:, n] - b[:, n]).max() <= 1e-6 * np.abs(b[:, n]).max()
    g.close()
    o.close()
