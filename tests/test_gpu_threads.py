"""Host threads that read one simulation's state at the same time."""
import threading

import pytest

pytestmark = pytest.mark.gpu


def test_threads_read_their_own_shape(cup):
    """Each reader gets the state of the shape it asked for, whoever else reads (a control loop
    and a logger, say): no value may differ from the one read alone."""
    shapes = [cup.disk(0.02 + 0.005 * k, 0.2 + 0.2 * k, 0.25, xvel=0.1 * k, bForced=True)
              for k in range(4)]
    sim = cup.Simulation(16, 8, extent=1.0, nu=1e-3, poisson="freespace", shapes=shapes)
    sim.reset()
    sim.simulate(3)
    alone = [sim.shape(k) for k in range(len(shapes))]
    time = sim.scalars()["time"]
    wrong = []

    def reader(k):
        for _ in range(300):
            if sim.shape(k) != alone[k] or sim.scalars()["time"] != time:
                wrong.append(k)

    threads = [threading.Thread(target=reader, args=(k,)) for k in range(len(shapes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    sim.close()
