"""The adjoint's buffers when the device cannot hold them."""
import pytest

pytestmark = pytest.mark.gpu


def test_adjoint_after_failed_allocation(cup):
    """A segment of 1e8 steps (130 TB) is refused, also when asked for again, and the simulation
    goes on: a run that fits gives the J of a simulation that never asked."""
    got = []
    for ask in (False, True):
        sim = cup.Simulation(8, 4, extent=1.0, nu=1e-3, CFL=0.1, poisson="freespace",
                             shapes=[cup.disk(0.06, 0.4, 0.25, xvel=0.2, bFixed=True,
                                              bForced=True)])
        sim.reset()
        sim.set_surface_velocity([0.01] * 8, 0)
        if ask:
            for _ in range(2):
                with pytest.raises(cup.Cup2dError) as e:
                    sim.adjoint_forward(2, every=100_000_000)
                assert e.value.code == cup.ERR_HIP
        got.append(sim.adjoint_forward(3, every=2)[0])
        sim.close()
    assert got[0] == got[1]
