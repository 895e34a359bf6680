"""The ghost remap of the conserved variables and the passive scalars, one launch
for both, against the oracle bit for bit: no scalar, one and the most a
configuration may have, both equations of state."""
import numpy as np
import pytest

from helpers import atm_config, sw_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx, nx1, ntracer, water", [
    (4, 3, 0, False), (4, 3, 1, False), (10, 7, 4, False), (18, 5, 3, False), (6, 1, 2, True),
    (12, 3, 4, True),
])
def test_ghosts_are_the_oracles(ex, orc, nx, nx1, ntracer, water):
    if water:
        cfg = sw_config(ex, nx=nx, nx1=nx1)
        cfg.ntracer = ntracer
    else:
        cfg = atm_config(ex, nx=nx, nx1=nx1, ntracer=ntracer)
    u0, _ = ex.init_state(cfg, 0 if water else 1, 7 * nx + ntracer)
    s0 = None
    if ntracer:
        s0 = np.random.default_rng(nx).random((6, ntracer) + u0.shape[2:]) * u0[:, :1]
    g, o = ex.Solver(cfg), orc.Oracle(cfg)
    for m in (g, o):
        m.upload(u0, s0)
        m.fill_ghosts()
    k = slice(3, 3 + nx)
    i = slice(3, 3 + nx1)
    pairs = list(zip(g.download(), o.download()))
    for a, b in pairs[:1 + bool(ntracer)]:
        for side in (slice(0, 3), slice(3 + nx, 6 + nx)):
            assert np.array_equal(a[:, :, k, side, i], b[:, :, k, side, i])
            assert np.array_equal(a[:, :, side, k, i], b[:, :, side, k, i])
    g.close()
    o.close()
