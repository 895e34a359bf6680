"""Infinities, NaNs and signed zeros beside a panel edge reach the neighbour's
ghost cells as the oracle's division hands them on (an infinity over a finite
divisor is that infinity), in the conserved variables and the passive scalars."""
import numpy as np
import pytest

from helpers import atm_config, sw_config

pytestmark = pytest.mark.gpu


def same(a, b):
    zero = (a == 0) & (b == 0)
    return np.array_equal(a, b, equal_nan=True) and \
        np.array_equal(np.signbit(a[zero]), np.signbit(b[zero]))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, -0.0])
@pytest.mark.parametrize("water", [True, False])
def test_ghosts_of_a_non_finite_state(ex, orc, water, value):
    nx, nx1 = 8, 4
    cfg = sw_config(ex, nx=nx, nx1=nx1) if water else atm_config(ex, nx=nx, nx1=nx1)
    cfg.ntracer = 2
    u0, _ = ex.init_state(cfg, 0 if water else 1, 5)
    s0 = np.random.default_rng(2).random((6, 2) + u0.shape[2:]) * u0[:, :1]
    rng = np.random.default_rng(9)
    for n in [0, 2, 3] if water else range(5):  # a few of each panel's cells
        hit = rng.random(u0[:, n].shape) < 0.1
        u0[:, n][hit] = value
    s0[rng.random(s0.shape) < 0.1] = value
    g, o = ex.Solver(cfg), orc.Oracle(cfg)
    for m in (g, o):
        m.upload(u0, s0)
        m.fill_ghosts()
    k, i = slice(3, 3 + nx), slice(3, 3 + nx1)
    for a, b in zip(g.download(), o.download()):
        for side in (slice(0, 3), slice(3 + nx, 6 + nx)):
            assert same(a[:, :, k, side, i], b[:, :, k, side, i])
            assert same(a[:, :, side, k, i], b[:, :, side, k, i])
    g.close()
    o.close()
