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
