"""Stencils on grids whose last strip of columns is ragged: bit-exact against the oracle (advDiff's
inner cells; the boundary cells carry a correction summed in another order, within 1e-15 of
values below one) and the numpy restatement (right-hand side and projection)."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
import numpy_ref as R  # noqa: E402

pytestmark = pytest.mark.gpu


# the last strip holds 32 cells (half a wave), 224, and all but 32 of its 256
@pytest.mark.parametrize("bp", [(9, 2), (15, 1), (23, 2), (63, 1), (5, 1)])
def test_ragged_strips_bitexact(cup, oracle_mod, bp):
    rng = np.random.default_rng(17)
    kw = dict(extent=1.0, nu=3e-3)
    g, o = cup.Simulation(*bp, **kw), oracle_mod.Oracle(*bp, **kw)
    vel = 0.3 * rng.standard_normal((2, g.NY, g.NX))
    for sim in (g, o):
        sim.set_field(0, vel)
        sim.set_scalars(uinf=(-0.11, 0.07))
        sim.advdiff(1.3e-3)
    a, b = g.get_field(cup.VEL), o.get_field(oracle_mod.VEL)
    inner = (slice(None), slice(1, -1), slice(1, -1))
    assert np.array_equal(a[inner], b[inner]) and np.abs(a - b).max() < 1e-15
    h, dt = g.scalars()["h"], 2e-3
    g.pressure_rhs(dt)
    assert np.array_equal(g.get_field(cup.TMP)[0], R.pressure_rhs(a[0], a[1], dt, h))
    p = rng.standard_normal((g.NY, g.NX))
    g.set_field(cup.PRES, p[None])
    g.pressure_correction(dt)
    u1, v1 = R.pressure_correction(a[0], a[1], p, dt, h)
    out = g.get_field(cup.VEL)
    assert np.array_equal(out[0], u1) and np.array_equal(out[1], v1)
    assert g.find_max_u() == np.abs(np.stack([u1 - 0.11, v1 + 0.07, u1, v1])).max()
