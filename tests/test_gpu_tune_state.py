"""Tuning leaves the time-step state alone: dt and the previous dt that bounds
the next step's growth, of a handle and of every member of a batch, when the
launches are timed and when an earlier result is taken over, and the step after
it is the untuned one's."""
import numpy as np
import pytest

from helpers import atm_config, sw_config

pytestmark = pytest.mark.gpu


def pair(ex, cfg):
    """two handles of one state, both bound to a small next step"""
    kind = 1 if cfg.eos == ex.EOS_IDEAL else 0
    u0, _ = ex.init_state(cfg, kind, 11)
    out = []
    for _ in range(2):
        g = ex.Solver(cfg)
        g.upload(u0)
        g.set_dt_state(0.5, 0.25)
        out.append(g)
    return out


def configs(ex):
    mixed = sw_config(ex, nx=10, nx1=1, rsolver=1)
    mixed.precision = ex.PREC_MIXED
    return [sw_config(ex, nx=12, nx1=1), mixed, atm_config(ex, nx=6, nx1=6)]


@pytest.mark.parametrize("which", [0, 1, 2])
def test_tuned_handle_keeps_its_time_step(ex, which):
    cfg = configs(ex)[which]
    cfg.cfl = 0.4 + which * 1e-3
    for _ in range(2):  # timed, then from the earlier result
        g, twin = pair(ex, cfg)
        g.tune(reps=2)
        assert g.dt_state() == (0.5, 0.25)
        assert g.step(1) == twin.step(1) == 0.5
        assert np.array_equal(g.download()[0], twin.download()[0])
        g.close()
        twin.close()


def test_tuned_batch_keeps_its_members_time_steps(ex):
    cfgs = configs(ex)
    for _ in range(2):
        pairs = [pair(ex, c) for c in cfgs]
        b = ex.Batch([p[0] for p in pairs])
        b.tune(reps=1)
        assert [p[0].dt_state() for p in pairs] == [(0.5, 0.25)] * len(pairs)
        b.step(1)
        for g, twin in pairs:
            assert twin.step(1) == 0.5
            assert g.dt_state() == twin.dt_state()
        b.close()
        for p in pairs:
            p[0].close()
            p[1].close()


@pytest.mark.parametrize("nx, mixed", [(34, False), (34, True), (128, False), (128, True)])
def test_tuning_between_and_after_shallow_water_stages(ex, nx, mixed):
    """the tuner repeats a fused stage and its halo: neither the stage register
    nor the state may see it, and the tuned step is the untuned one's"""
    cfg = sw_config(ex, nx=nx, nx1=2, rsolver=1)
    cfg.precision = ex.PREC_MIXED if mixed else ex.PREC_FP64
    g, twin = pair(ex, cfg)
    for stage in (1, 2, 3):
        g.tune(reps=1)
        for m in (g, twin):
            m.stage(stage, 2.0)
    widths = g.tune(reps=1)
    assert set(ex.LAUNCH_KINDS) <= set(widths)
    assert g.step(3) == twin.step(3)
    assert np.array_equal(g.download()[0], twin.download()[0])
    assert np.array_equal(g.prim(), twin.prim())
    g.close()
    twin.close()
    b = ex.Batch([pair(ex, cfg)[0], pair(ex, cfg)[0]])
    b.set_caps({"sw_stage": 300, "sw_stage_mix": 300, "sw_halo": 5, "sw_edge": 3, "dt": 9})
    b.step(2)
    g = pair(ex, cfg)[0]
    g.step(2)
    for m in b.members:
        assert np.array_equal(m.download()[0], g.download()[0])
    b.close()
