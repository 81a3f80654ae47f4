"""Networks of no neurons: alone in a simulation they step (nothing is
launched), beside others they change nothing."""
import numpy as np
import pytest

import neurocorrelation_amd as nc
from neurocorrelation_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [{}, dict(waves_per_block=2), dict(waves_per_block=2, graph_steps=4),
                                   dict(waves_per_block=4, persistent=1)])
def test_only_empty_networks(shape):
    net = nc.Network.from_edges(0, [], [], [], [])
    sim = nc.Simulation(64, 64, 2)
    a, b = sim.add(net), sim.add(net, steps=7)
    sim.set_launch(**shape)
    for steps in (1, 20, 20):
        sim.step(steps)
        sim.synchronize()
    assert sim.progress(a)[0] == 41 and sim.progress(b) == (7, 0)
    assert sim.potential(a, 0).size == 0
    saved = sim.save(a)
    sim.close()
    other = nc.Simulation(64, 64, 1)
    c = other.add(net)
    other.restore(c, saved)
    assert other.progress(c)[0] == 41
    other.close()


@pytest.mark.parametrize("n", [100, 1500])
def test_an_empty_network_beside_another(n):
    net = nc.Network.generate(n, W.side_for(n), W.radius_for_degree(20), 1, 20, seed=1)
    states = []
    for empty in (False, True):
        sim = nc.Simulation(n + 128, net.n_syn + 64, 3)
        if empty:
            sim.add(nc.Network.from_edges(0, [], [], [], []))
        i = sim.add(net)
        sim.push_forced(i, np.arange(1, 21), np.arange(20), np.zeros(20))
        sim.step(40)
        first = sim.save(i)
        if empty:  # the neurons go, the empty network stays, the neurons come again
            sim.remove(i)
            sim.step(3)
            i = sim.add(net)
            sim.restore(i, first)
        sim.step(30)
        states.append((first, sim.save(i)))
        sim.close()
    assert states[0] == states[1]
