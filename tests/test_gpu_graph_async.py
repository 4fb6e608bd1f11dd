"""Captured steps enqueued without waiting in between, so that a graph is replaced while its
launches run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def member(cup, k):
    sim = cup.Simulation(16, 8, extent=1.0, nu=1e-4, CFL=0.1, poisson="freespace",
                         shapes=[cup.disk(0.04 + 0.01 * k, 0.3, 0.25, xvel=0.2, bFixed=True,
                                          bForced=True)])
    sim.reset()
    sim.set_field(cup.VEL, 0.02 * np.random.default_rng(k).standard_normal((2, sim.NY, sim.NX)))
    return sim


def state(cup, sim):
    return (sim.get_field(cup.VEL).tobytes(), sim.get_field(cup.PRES).tobytes(),
            sorted(sim.shape().items()), sorted(sim.scalars().items()))


def test_ensemble_recaptured_in_flight(cup):
    """An odd number of steps and another number of lanes each need new graphs: no wait by the
    caller, and each member equals the one advanced alone."""
    alone, members = ([member(cup, k) for k in range(3)] for _ in range(2))
    ens = cup.Ensemble(members)
    ens.simulate(5, sync=False)
    ens.simulate(4, sync=False)
    ens.set_lanes(3)
    ens.simulate(6, sync=False)
    ens.set_lanes(2)
    ens.simulate(4)
    for sim in alone:
        sim.simulate(19)
    for a, b in zip(alone, members):
        assert state(cup, a) == state(cup, b)
    ens.close()


def test_graphs_of_both_parities_in_flight(cup):
    a, b = member(cup, 0), member(cup, 0)
    for n in (4, 3, 2, 5):
        a.simulate_graph(n, sync=False)
        a.simulate(1, sync=False)
    b.simulate(18)
    assert state(cup, a) == state(cup, b)
