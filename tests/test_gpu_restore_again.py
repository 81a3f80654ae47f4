"""A checkpoint taken before its first step, with spikes in flight, restored
into the same network twice: the network is as after one restore, and so is
the network whose slots lie behind its own.  Rows are whole (every slot of a
slice holds a synapse), so that lists that held every spike twice would not
fit their slices."""
import numpy as np
import pytest

import neurocorrelation_amd as nc

pytestmark = pytest.mark.gpu

HEADER = 56  # bytes before the neurons; 12 bytes a neuron, 16 a synapse (weight, depolarisation, last arrival, arrival)


def _rows(n, k, seed):
    rng = np.random.default_rng(seed)
    to = np.repeat(np.arange(n), k)
    frm = np.concatenate([(t + 1 + rng.choice(n - 1, k, replace=False)) % n for t in range(n)])
    return nc.Network.from_edges(n, to, frm, rng.uniform(0.1, 0.6, n * k).astype(np.float32),
                                 rng.integers(1, 100, n * k).astype(np.uint8))


def _in_flight(fresh, n, arrivals):
    b = bytearray(fresh)
    syn = np.frombuffer(b, np.int32, offset=HEADER + 12 * n).reshape(-1, 4)
    syn[:, 3] = arrivals
    syn[:, 1] = np.full(len(syn), 3.5, np.float32).view(np.int32)
    return bytes(b)


# arrivals in one window's list, in both, and in the other from the first time
@pytest.mark.parametrize("n,k", [(64, 8), (130, 16), (1500, 24)])
@pytest.mark.parametrize("spread", [1, 40, 255])
def test_restored_twice_is_restored_once(n, k, spread):
    net, behind = _rows(n, k, 1), _rows(70, 8, 2)
    first = 1 + np.arange(net.n_syn) % spread
    states = []
    for twice in (False, True):
        sim = nc.Simulation(n + 64 + 128, net.n_syn + behind.n_syn, 2,
                            max_slots=net.device_size()[1] + behind.device_size()[1])
        a, b = sim.add(net), sim.add(behind)
        fresh, fresh_b = sim.save(a), sim.save(b)
        sim.restore(b, _in_flight(fresh_b, 70, 1 + np.arange(behind.n_syn) % 30))
        if twice:
            sim.restore(a, _in_flight(fresh, n, first + (16 if spread == 1 else 0)))
        sim.restore(a, _in_flight(fresh, n, first))
        out = [sim.save(a), sim.save(b)]
        for steps in (1, 30, 260):
            sim.step(steps)
            out += [sim.save(a), sim.save(b)]
        states.append(out)
        sim.close()
    assert states[0] == states[1]
    assert any(states[0][2 * i] != states[0][0] for i in range(1, 4))
