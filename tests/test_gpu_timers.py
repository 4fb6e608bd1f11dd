"""The named timers of runs with disks only, whose steps otherwise take several parts per launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SINGLE = ("put_objects", "advdiff", "rhs_obstacles", "fade", "forces", "penalize")
ITERATIVE = ("put_objects", "advdiff", "flux_fix", "forces")


def simulation(cup, poisson, iterative):
    sim = cup.Simulation(9, 5, extent=1.0, nu=1e-3, CFL=0.1, poisson=poisson, fadeLen=0.02,
                         iterative_penal=iterative,
                         shapes=[cup.disk(0.06, 0.4, 0.28, xvel=0.2, bFixed=True, bForced=True),
                                 cup.disk(0.03, 0.7, 0.28)])
    sim.reset()
    return sim


def state(cup, sim):
    return ([sim.get_field(f).tobytes() for f in (cup.VEL, cup.PRES, cup.CHI)]
            + [sorted(sim.shape(k).items()) for k in range(2)] + [sorted(sim.scalars().items())])


@pytest.mark.parametrize("poisson,iterative", [("freespace", False), ("freespace", True)])
@pytest.mark.parametrize("every", [1, 3])
def test_disk_step_timers(cup, poisson, iterative, every):
    """Each part of a step is one launch under its own name (every k-th one with sampling), and
    timing changes no bit of the result."""
    n = 9
    plain, timed = (simulation(cup, poisson, iterative) for _ in range(2))
    timed.timer_sample("*", every)
    timed.timer_enable("*", 4 * n)
    for sim in (plain, timed):
        sim.simulate(n)
    for name in ITERATIVE if iterative else SINGLE:
        ms, launches = timed.timer_read(name)
        assert launches == n // every and ms > 0, (name, launches, ms)
    timed.timer_enable("*", 0)
    for sim in (plain, timed):
        sim.simulate(2)
    assert state(cup, plain) == state(cup, timed)


def test_timed_adjoint(cup):
    """The adjoint's runs with a part timed: the same J, time steps and gradient."""
    theta = 0.02 * np.random.default_rng(3).standard_normal(16)
    got = []
    for timed in (False, True):
        sim = cup.Simulation(8, 4, extent=1.0, nu=1e-3, CFL=0.1, poisson="freespace",
                             shapes=[cup.disk(0.06, 0.4, 0.25, xvel=0.2, bFixed=True,
                                              bForced=True)])
        sim.reset()
        sim.set_surface_velocity(theta, 0)
        if timed:
            sim.timer_enable("forces", 64)
        J, dts = sim.adjoint_forward(7, every=3)
        if timed:
            assert sim.timer_read("forces")[1] == 7
        g = sim.adjoint_backward()
        got.append((J, dts, g))
    # (the drag's scatter adds in any order: the gradients agree to rounding)
    assert got[0][0] == got[1][0] and np.array_equal(got[0][1], got[1][1])
    assert np.linalg.norm(got[0][2] - got[1][2]) <= 1e-12 * np.linalg.norm(got[0][2])
