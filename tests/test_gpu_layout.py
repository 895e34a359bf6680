"""Host transfers through the device's layout kernel: a random state (every
ghost and corner cell a value of its own) comes back bit for bit where nothing
rewrites it, at sizes on and around the 32 x 32 tiles and with more planes than
one staged piece.  The upload rewrites only the x2 / x3 ghost strips of interior
levels (the ghost fill)."""
import numpy as np
import pytest

from helpers import atm_config, sw_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eos, nx, nx1, ntracer", [
    ("sw", 4, 1, 0),     # the smallest panel
    ("sw", 26, 3, 0),    # nc2 = 32, one tile
    ("air", 28, 26, 1),  # nc2 = 34, nc1 = 32
    ("air", 26, 27, 3),  # nc2 = 32, nc1 = 33
    ("air", 64, 59, 2),  # 70 x 65 planes, 2100 of them: several pieces, the last one partial
])
def test_state_round_trip(ex, eos, nx, nx1, ntracer):
    cfg = sw_config(ex, nx=nx, nx1=nx1) if eos == "sw" else \
        atm_config(ex, nx=nx, nx1=nx1, ntracer=ntracer)
    u0, s0 = ex.init_state(cfg, 0 if eos == "sw" else 1, 3)
    rng = np.random.default_rng(nx + nx1)
    keep = np.ones(u0.shape[2:], bool)  # cells no ghost fill writes
    side, lev = slice(3, -3), slice(3, 3 + nx1)
    keep[:3, side, lev] = keep[-3:, side, lev] = False
    keep[side, :3, lev] = keep[side, -3:, lev] = False
    inner = np.zeros_like(keep)
    inner[side, side, lev] = True
    u0[:, :, ~inner] = rng.random(u0[:, :, ~inner].shape)
    if s0 is not None:
        s0[:] = rng.random(s0.shape)
    g = ex.Solver(cfg)
    g.upload(u0, s0)
    u, s = g.download()
    assert np.array_equal(u[:, :, keep], u0[:, :, keep])
    if s0 is not None:
        assert np.array_equal(s[:, :, keep], s0[:, :, keep])
    w = g.prim()  # the third array that comes back: density is the conserved one
    assert np.array_equal(w[:, 0][:, inner], u0[:, 0][:, inner])
    g.close()
