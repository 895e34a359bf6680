"""What a step of shallow water without scalars leaves for the calls that
follow it, against the oracle: the last stage's face fluxes and the stage
register (the step's first state), after an eager step, replayed ones, a redone
loop and a batch, on panels with one tile and with several; and a step whose
primitive state is older than its conserved one (no ghost fill between), which
takes its first fluxes from the primitive state."""
import numpy as np
import pytest

from helpers import interior, sw_config

pytestmark = pytest.mark.gpu


def pair(ex, orc, nx, nx1, solver):
    cfg = sw_config(ex, nx=nx, nx1=nx1, rsolver=solver)
    u0, _ = ex.init_state(cfg, 0, 3 * nx + solver)
    g, o = ex.Solver(cfg), orc.Oracle(cfg)
    for m in (g, o):
        m.upload(u0)
    return g, o


def same_fluxes(g, o, nx, nx1):
    s, f, i = slice(3, 3 + nx), slice(3, 4 + nx), slice(3, 3 + nx1)
    a, b = g.flux(1), o.flux(1)
    for n in (0, 2, 3):
        assert np.array_equal(a[:, n, s, f, i], b[:, n, s, f, i]), n
    a, b = g.flux(2), o.flux(2)
    for n in (0, 2, 3):
        assert np.array_equal(a[:, n, f, s, i], b[:, n, f, s, i]), n


SIZES = [(4, 1, 0), (16, 1, 1), (34, 2, 0), (64, 3, 1)]


@pytest.mark.parametrize("how", ["one", "many", "given", "redo", "batch", "graph"])
@pytest.mark.parametrize("nx, nx1, solver", SIZES)
def test_fluxes_and_register_of_the_last_stage(ex, orc, nx, nx1, solver, how):
    g, o = pair(ex, orc, nx, nx1, solver)
    if how == "one":
        assert g.step(1) == o.step(1)
    elif how == "many":
        assert g.step(3) == o.step(3)
    elif how == "given":
        g.step(2, 40.0)
        o.step(2, 40.0)
    elif how == "redo":
        g.step_redo(2, 1)
        o.step(2)
    else:
        b = ex.Batch([g], graph=how == "graph")
        b.step(2)
        b.step(1)
        b.close()
        o.step(3)
    same_fluxes(g, o, nx, nx1)
    # stage 2 from these fluxes and the register
    dt = 30.0
    g.integrate_hydro(2, dt)
    o.add_flux_divergence(0.25 * dt, 2)
    assert np.array_equal(interior(g.download()[0], nx1), interior(o.download()[0], nx1))
    g.close()
    o.close()


@pytest.mark.parametrize("nx, solver", [(8, 0), (34, 1), (128, 0)])
def test_mixed_fluxes_of_the_last_stage(ex, nx, solver):
    """the mixed form's fluxes are seen through the update they make: equal to
    those exo_stage leaves, bit for bit"""
    cfg = sw_config(ex, nx=nx, nx1=1, rsolver=solver)
    cfg.precision = ex.PREC_MIXED
    u0, _ = ex.init_state(cfg, 0, nx)
    g, f = ex.Solver(cfg), ex.Solver(cfg)
    for m in (g, f):
        m.upload(u0)
    dt = g.step(1, 20.0)
    for stage in (1, 2, 3):
        f.stage(stage, dt)
    for m in (g, f):
        m.integrate_hydro(3, dt)
    assert np.array_equal(interior(g.download()[0], 1), interior(f.download()[0], 1))
    g.close()
    f.close()


@pytest.mark.parametrize("nx, nx1, solver", SIZES)
def test_step_with_an_older_primitive_state(ex, orc, nx, nx1, solver):
    g, o = pair(ex, orc, nx, nx1, solver)
    for m in (g, o):
        m.calc_fluxes()
        m.add_flux_divergence(60.0)  # into u; w is left to the ghost fill
    assert g.step(1, 20.0) == o.step(1, 20.0)
    assert np.array_equal(interior(g.download()[0], nx1), interior(o.download()[0], nx1))
    g.close()
    o.close()
