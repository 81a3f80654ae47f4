"""State read, written and checkpointed on the device, in the caller's orders:
against each other and against the documented byte layout of a checkpoint, at
sizes below and above what goes through pinned memory (1 MiB), for rows of 0,
1, 15-17 and many synapses."""
import numpy as np
import pytest

import neurocorrelation_amd as nc
from neurocorrelation_amd import workloads as W

pytestmark = pytest.mark.gpu


def _rows(degrees, seed):
    """A network whose neuron t has degrees[t] incoming synapses."""
    rng = np.random.default_rng(seed)
    n = len(degrees)
    to, frm = [], []
    for t, d in enumerate(degrees):
        src = rng.choice(n - 1, d, replace=False)
        frm.append(src + (src >= t))
        to.append(np.full(d, t))
    to, frm = np.concatenate(to), np.concatenate(frm)
    w = rng.uniform(-0.5, 0.5, len(to)).astype(np.float32)
    return nc.Network.from_edges(n, to, frm, w, rng.integers(1, 100, len(to)).astype(np.uint8))


def _made(kind):
    if kind == "rows":
        return _rows([0, 1, 15, 16, 17, 31, 33, 200] * 40, 1)
    n = {"small": 500, "large": 9000}[kind]
    return nc.Network.generate(n, W.side_for(n), W.radius_for_degree(60), 1, 90, 0.2, 0.8, 0.1, seed=2)


def _running(net):
    sim = nc.Simulation(net.n + 256, net.n_syn + 4096, 2)
    sim.add(_rows([3] * 70, 5))  # the network's positions, slots and edges start past another's
    drive = W.drive_spec(dict(n_inputs=net.n // 4, n_groups=2, n_correlated=4, period=50, p0=0.2, amp_corr=1.0,
                              amp_ind=1.0, bg_prob=0.01), seed=4)
    nid = sim.add(net, None, drive)
    sim.step(150)
    return sim, nid


@pytest.mark.parametrize("kind", ["rows", "small", "large"])
def test_reads_agree_with_the_checkpoint(kind):
    net = _made(kind)
    sim, nid = _running(net)
    n, S = net.n, net.n_syn
    raw = np.frombuffer(sim.save(nid), np.uint8)[56:]
    neurons = raw[:12 * n].view(np.uint32).reshape(n, 3)
    syn = raw[12 * n:12 * n + 16 * S].view(np.uint32).reshape(S, 4)
    assert np.array_equal(neurons[:, 0], sim.potential(nid, n).view(np.uint32))
    assert np.array_equal(neurons[:, 1], sim.last_fire(nid, n).view(np.uint32))
    assert np.array_equal(neurons[:, 2], sim.firings(nid, n))
    assert np.array_equal(syn[:, 0], sim.weights(nid, S).view(np.uint32))
    arrival, last, depol = sim.synapse_state(nid, S)
    arr = syn[:, 3].view(np.int32)
    assert np.array_equal(syn[:, 1], depol.view(np.uint32))
    assert np.array_equal(syn[:, 2], last.view(np.uint32))
    held = (arr != nc.NEVER) & (150 < arr + 3)  # a release window of 3 steps at 1 ms
    assert np.array_equal(arrival, np.where(held, arr, 0))
    assert held.any() and (last != nc.NEVER).any()
    for m in (0, 1, 7, S // 2 + 1):  # the first m
        assert np.array_equal(sim.weights(nid, m), sim.weights(nid, S)[:m])
        assert all(np.array_equal(x, y[:m]) for x, y in zip(sim.synapse_state(nid, m), (arrival, last, depol)))
    assert np.array_equal(sim.potential(nid, 5), sim.potential(nid, n)[:5])
    sim.close()


@pytest.mark.parametrize("kind", ["rows", "small", "large"])
def test_weights_written_and_edited(kind):
    net = _made(kind)
    sim, nid = _running(net)
    S = net.n_syn
    rng = np.random.default_rng(3)
    want = rng.uniform(-1, 1, S).astype(np.float32)
    sim.write_weights(nid, want)
    assert np.array_equal(sim.weights(nid, S), want)
    part = rng.uniform(-1, 1, S // 3 + 1).astype(np.float32)
    sim.write_weights(nid, part)
    want[:len(part)] = part
    assert np.array_equal(sim.weights(nid, S), want)
    # unordered, with repeats (the last of each holds), the first and the last synapse
    syn = np.concatenate([rng.integers(0, S, 300), [S - 1, 0, 5, 5, 5]])
    w = rng.uniform(-1, 1, len(syn)).astype(np.float32)
    sim.set_weights(nid, syn, w)
    for k, x in zip(syn, w):
        want[k] = x
    assert np.array_equal(sim.weights(nid, S), want)
    # more entries than synapses
    syn = rng.integers(0, min(S, 1000), 3000)
    w = rng.uniform(-1, 1, 3000).astype(np.float32)
    sim.set_weights(nid, syn, w)
    for k, x in zip(syn, w):
        want[k] = x
    assert np.array_equal(sim.weights(nid, S), want)
    sim.close()


@pytest.mark.parametrize("kind", ["rows", "small", "large"])
def test_a_restored_network_continues(kind):
    net = _made(kind)
    sim, nid = _running(net)
    saved = sim.save(nid)
    drive = W.drive_spec(dict(n_inputs=net.n // 4, n_groups=2, n_correlated=4, period=50, p0=0.2, amp_corr=1.0,
                              amp_ind=1.0, bg_prob=0.01), seed=4)
    other = nc.Simulation(net.n + 64, net.n_syn)
    oid = other.add(net, None, drive)
    other.restore(oid, saved)
    assert other.save(oid) == saved
    for steps in (1, 120):
        sim.step(steps)
        other.step(steps)
        assert sim.save(nid) == other.save(oid)
    sim.close()
    other.close()
