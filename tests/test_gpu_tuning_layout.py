"""A tuning result kept by a caller as the C entry points lay it out: 30 widths,
then 30 shapes from index EXO_NKINDS on, taken back by exo_batch_set_caps as it
was given out, also where a caller's array ends there."""
import ctypes as C

import numpy as np
import pytest

from helpers import atm_config, interior, sw_config

pytestmark = pytest.mark.gpu


def test_sixty_values_are_widths_then_shapes(ex):
    cfg = atm_config(ex, nx=6, nx1=6)
    u0, _ = ex.init_state(cfg, 1, 3)
    g, twin = ex.Solver(cfg), ex.Solver(cfg)
    for m in (g, twin):
        m.upload(u0)
    b = ex.Batch([g])
    kept = np.zeros(60, dtype=np.int32)
    kept[0] = 7                                    # a width: the conversion
    kept[30 + 3], kept[30 + 4] = 8, 2              # shapes: both forms' x1 sweeps
    assert b.L.exo_batch_set_caps(b.h, kept.ctypes.data_as(C.c_void_p), len(kept)) == 0
    b.step(2)
    twin.step(2)
    assert np.array_equal(interior(g.download()[0], 6), interior(twin.download()[0], 6))
    out = np.full(60, -1, dtype=np.int32)
    assert b.L.exo_batch_tune(b.h, 1, out.ctypes.data_as(C.c_void_p), len(out)) == 0
    assert np.all(out >= 0)
    # every shape but the x1 sweeps' is the default
    assert not out[30:33].any() and not out[35:].any()
    assert b.L.exo_batch_set_caps(b.h, out.ctypes.data_as(C.c_void_p), len(out)) == 0
    b.close()
    g.close()
    twin.close()


def test_kinds_added_later_follow_the_shapes(ex):
    """the whole array, given out and taken back, and its last four values"""
    cfg = sw_config(ex, nx=34, nx1=1)
    u0, _ = ex.init_state(cfg, 0, 3)
    g, twin = ex.Solver(cfg), ex.Solver(cfg)
    for m in (g, twin):
        m.upload(u0)
    b = ex.Batch([g])
    b.tune(1)
    kept = np.full(64, -1, dtype=np.int32)
    assert b.L.exo_batch_tune(b.h, 1, kept.ctypes.data_as(C.c_void_p), len(kept)) == 0
    assert np.all(kept >= 0)
    kept[60:] = 3, 3, 2, 1
    assert b.L.exo_batch_set_caps(b.h, kept.ctypes.data_as(C.c_void_p), len(kept)) == 0
    b.step(2)
    twin.step(2)
    assert np.array_equal(interior(g.download()[0], 1), interior(twin.download()[0], 1))
    assert ex.LAUNCH_KINDS[30:] == ("sw_stage", "sw_stage_mix", "sw_halo", "sw_edge")
    b.close()
    g.close()
    twin.close()
