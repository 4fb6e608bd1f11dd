"""ComputeForces called by itself, with no body update before it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("placed", [False, True])
def test_compute_forces_without_body_update(cup, oracle_mod, placed):
    """Right after reset, and after the bodies were placed again: the forces are those of the
    bodies' present state (ComputeForces.cpp:16-111), within the whole-step bound of 1e-8 for the
    drag; torques about a centre shifted by a step would be off by a percent."""
    def shapes(m):
        return [m.disk(0.07, 0.35, 0.25, xvel=0.3, yvel=-0.1, bForced=True),
                m.disk(0.05, 0.7, 0.3, xvel=-0.2, bForced=True)]
    rng = np.random.default_rng(31)
    kw = dict(extent=1.0, nu=1e-2, CFL=0.1, poisson="freespace")
    used = cup.Simulation(8, 4, shapes=shapes(cup), **kw)  # leaves its state in the memory reused
    used.reset()
    used.simulate(3)
    used.close()
    g, o = cup.Simulation(8, 4, shapes=shapes(cup), **kw), oracle_mod.Oracle(8, 4, shapes=shapes(oracle_mod), **kw)
    vel = 0.3 * rng.standard_normal((2, g.NY, g.NX))
    pres = rng.standard_normal((g.NY, g.NX))
    for sim in (g, o):
        sim.reset()
        if placed:
            sim.put_objects(0.02)
        sim.set_field(0, vel)
        sim.set_field(2, pres[None])
        sim.compute_forces()
    for k in range(2):
        a, b = g.shape(k), o.shape(k)
        scale = np.hypot(b["forcex"], b["forcey"])
        for key in ("forcex", "forcey", "torque", "drag", "thrust", "Pthrust", "Pdrag", "perimeter"):
            assert abs(a[key] - b[key]) <= 1e-8 * max(scale, abs(b[key])), (k, key, a[key], b[key])
