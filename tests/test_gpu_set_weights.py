"""nc_set_weights on lists of every length and order, with repeats (the last
weight of a synapse holds), around where it takes them another way: a single
entry, ascending lists, short ones, those of more than a 256th of the synapses
and those of all."""
import numpy as np
import pytest

import neurocorrelation_amd as nc
from neurocorrelation_amd import workloads as W

pytestmark = pytest.mark.gpu


# in-degrees near 40, and rows of none between rows of many
@pytest.mark.parametrize("kind", ["job", "rows"])
def test_lists(kind):
    rng = np.random.default_rng(1)
    if kind == "job":
        net = nc.Network.generate(2000, W.side_for(2000), W.radius_for_degree(40), 1, 20, seed=1)
    else:
        deg = np.where(np.arange(900) % 7 == 3, 180, np.where(np.arange(900) < 40, 1, 0))
        to = np.repeat(np.arange(900), deg)
        frm = np.concatenate([(t + 1 + rng.choice(899, d, replace=False)) % 900 for t, d in enumerate(deg)])
        net = nc.Network.from_edges(900, to, frm, rng.uniform(0.1, 0.5, to.size).astype(np.float32),
                                    np.ones(to.size, np.uint8))
    S = net.n_syn
    sim = nc.Simulation(net.n + 64 + 128, S + 1000, 2)
    sim.add(nc.Network.from_edges(70, [1, 2], [0, 0], [0.5, 0.5], [1, 1]))
    i = sim.add(net)
    want = sim.weights(i, S)
    line = S // 256
    for m in (1, 2, line - 1, line, line + 1, 5 * line, S // 2, S, 2 * S):
        for order in ("ascending", "shuffled", "descending", "repeated"):
            if order == "repeated":
                syn = rng.integers(0, max(1, min(S, m // 2 + 1)), m)
            elif m > S:
                continue
            else:
                syn = rng.choice(S, m, replace=False)
                syn = {"ascending": np.sort(syn), "descending": np.sort(syn)[::-1]}.get(order, syn)
            w = rng.uniform(-1, 1, m).astype(np.float32)
            sim.set_weights(i, syn, w)
            for k, x in zip(syn, w):
                want[k] = x
            assert np.array_equal(sim.weights(i, S), want), (m, order)
    with pytest.raises(nc.NCError):
        sim.set_weights(i, np.array([0, S]), np.ones(2, np.float32))
    assert np.array_equal(sim.weights(i, S), want)
    sim.close()
