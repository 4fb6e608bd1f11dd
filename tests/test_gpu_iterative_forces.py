"""Forces of whole steps with the iterative penalization and a swimmer, whose ComputeForces runs on
another stream beside the next step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def simulation(cup):
    sim = cup.Simulation(16, 16, extent=1.0, nu=1e-3, CFL=0.1, poisson="freespace",
                         iterative_penal=True,
                         shapes=[cup.carlingfish(0.5, 0.6, L=0.2, T=1.0),
                                 cup.disk(0.06, 0.4, 0.25, xvel=0.2, bForced=True)])
    sim.reset()
    sim.set_field(cup.VEL, 0.05 * np.random.default_rng(7).standard_normal((2, sim.NY, sim.NX)))
    sim.force_log_enable(16)
    return sim


def test_forces_do_not_depend_on_the_overlap(cup):
    """The force records of steps enqueued one behind the other are those of steps that are waited
    for one by one (then every ComputeForces has the device to itself), bit for bit, every time."""
    one = simulation(cup)
    for _ in range(6):
        one.simulate(1)
    want = [one.force_log(k).tobytes() for k in range(2)]
    for _ in range(5):
        sim = simulation(cup)
        sim.simulate(6)
        assert [sim.force_log(k).tobytes() for k in range(2)] == want
        sim.close()
