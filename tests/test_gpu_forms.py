"""The forms of the step kernels that the default launch shape chooses among
(a workgroup per network, several waves per slice) against the per-slice
kernels of an explicit launch shape, bit for bit: both take the same network
through the same steps.  The per-slice kernels equal the oracle
(test_gpu_parity.py), as does the default shape at its sizes."""
import numpy as np
import pytest

import neurocorrelation_amd as nc
from neurocorrelation_amd import workloads as W

pytestmark = pytest.mark.gpu

PER_SLICE = dict(waves_per_block=2)


def _net(n, k, delay_max=20, seed=1, inhib=0.0, w=(0.2, 0.8)):
    return nc.Network.generate(n, W.side_for(n), W.radius_for_degree(k), 1, delay_max, w[0], w[1], inhib, seed=seed)


def _drive(n, seed, bg=0.0):
    n_in = min(n, max(6, n // 20))
    return W.drive_spec(dict(n_inputs=n_in, n_groups=min(2, n_in), n_correlated=min(2, n_in), period=200, p0=0.05,
                             amp_corr=1.0, amp_ind=0.5, bg_prob=bg), seed=seed)


def _state(sim, nid, net, cap=0):
    out = [sim.potential(nid, net.n), sim.last_fire(nid, net.n), sim.firings(nid, net.n),
           sim.weights(nid, net.n_syn), np.frombuffer(sim.save(nid), np.uint8)]
    out += list(sim.synapse_state(nid, net.n_syn))
    if cap:
        out += list(sim.raster(nid, cap))
    return out


def _same(a, b):
    assert len(a) == len(b)
    for i, (x, y) in enumerate(zip(a, b)):
        assert x.shape == y.shape and np.array_equal(x.view(np.uint8), y.view(np.uint8)), "array %d differs" % i


def _both(net, drive, dt, calls, cap=1 << 20, events=None):
    """The network under both, each call's steps in turn; then each continues
    a few steps in the other's form (what one leaves has to serve the other)."""
    states = []
    for first, then in (({}, PER_SLICE), (PER_SLICE, {})):
        sim = nc.Simulation.for_network(net, raster_capacity=cap)
        nid = sim.add(net, nc.default_params(dt=dt), drive)
        sim.set_launch(**first)
        got = []
        for i, steps in enumerate(calls):
            if events:
                sim.push_forced(nid, *events(i, steps))
            if i == 1:
                sim.write_weights(nid, sim.weights(nid, net.n_syn) * np.float32(0.9))
            sim.step(steps)
            got += _state(sim, nid, net, cap)
        sim.set_launch(**then)
        sim.step(20)
        states.append(got + _state(sim, nid, net, cap))
        sim.close()
    _same(*states)


# one lane, a slice and its neighbours, the edges of the three group sizes
# (4, 8 and 16 slices), the first size past them, and more than a few
# workgroups; in-degrees within one mask word, across several, and past the
# forms' 256
@pytest.mark.parametrize("n,k", [(1, 4), (64, 10), (65, 40), (256, 30), (257, 60), (512, 50), (513, 20), (1024, 50),
                                 (1025, 50), (300, 4.24), (400, 330), (3000, 90)])
def test_sizes(n, k):
    net = _net(n, k, seed=n)
    _both(net, _drive(n, seed=n), 1.0, [60, 1, 40])


@pytest.mark.parametrize("dt", [1.0, 0.25, 1.0 / 16])
def test_steps_delays_and_background(dt):
    # delays past the buckets' 64 steps (pending lists), background fires,
    # calls longer than the drive ring; at 1/16 ms a trace table is longer
    # than the workgroup-per-network form stages
    net = _net(700, 40, delay_max=200, seed=3, inhib=0.2, w=(0.05, 0.3))
    _both(net, _drive(700, seed=3, bg=0.02), dt, [1100, 7, 90])


def test_host_events():
    net = _net(750, 12, seed=4)

    def events(i, steps):
        rng = np.random.default_rng(i)
        m = 300 if i else 5
        return rng.integers(1, steps + 4, m), rng.integers(0, 750, m), rng.integers(0, 2, m)
    _both(net, None, 0.5, [8, 8, 30], events=events)


def test_bucket_overflow():
    # 320 spikes into one slice at one step: past a bucket's 128 entries, and
    # more arrivals per lane than the group forms hand over
    src = np.arange(64, 64 + 320)
    to = np.repeat(np.arange(8), 40)
    net = nc.Network.from_edges(400, to, src, np.full(320, 0.4, np.float32), np.full(320, 9, np.uint8))

    def events(i, steps):
        return np.ones(320), src, np.zeros(320)
    _both(net, None, 1.0, [12, 12, 12], events=events)


def test_uneven_budgets():
    # networks of one simulation that stop at their own step counts, some
    # between calls, one with no synapse
    nets = [_net(n, 20, seed=n) for n in (70, 300, 900, 128)]
    nets.append(nc.Network.from_edges(3, [], [], [], []))
    steps = [30, 0, 75, 55, 10]
    got = []
    for shape in ({}, PER_SLICE):
        sim = nc.Simulation(4096, 200_000, 8, raster_capacity=1 << 18)
        ids = [sim.add(net, None, _drive(net.n, 5) if net.n > 3 else None, steps=s) for net, s in zip(nets, steps)]
        sim.set_launch(**shape)
        for c in (20, 40, 40):
            sim.step(c)
        got.append([x for i, net in zip(ids, nets) for x in _state(sim, i, net, 1 << 18)])
        sim.close()
    _same(*got)


def test_quiet_many_slices():
    # more than 8192 slices, which the default shape takes in XCD order
    net = nc.Network.generate(530_000, W.side_for(530_000), W.radius_for_degree(8), 1, 20, 0.05, 0.3, 0.2, seed=2,
                              device=0)
    _both(net, _drive(530_000, seed=2, bg=0.01), 1.0, [30, 30], cap=1 << 21)


# busy simulations of more than 1024 and more than 4096 slices, in networks of
# more than 16: two waves and one wave per slice, from the second call on (the
# first one's activity is read back with its state)
@pytest.mark.parametrize("n,nets", [(1500, 48), (30_000, 10)])
def test_busy_many_slices(n, nets):
    made = [nc.Network.generate(n + 37 * i, W.side_for(n), W.radius_for_degree(25), 1, 20, 0.2, 0.8, seed=i, device=0)
            for i in range(nets)]
    got = []
    for shape in ({}, PER_SLICE):
        sim = nc.Simulation(sum(m.n + 64 for m in made), sum(m.n_syn for m in made), nets)
        ids = [sim.add(m, None, _drive(m.n, i)) for i, m in enumerate(made)]
        sim.set_launch(**shape)
        out = []
        for c in (60, 20, 20):
            sim.step(c)
            out += [x for i, m in zip(ids, made) for x in (sim.potential(i, m.n), sim.firings(i, m.n))]
        out += [x for i, m in zip(ids[:3], made[:3]) for x in _state(sim, i, m)]
        got.append(out)
        sim.close()
    _same(*got)


def test_own_graphs_from_the_second_equal_call():
    # 3000 quiet neurons: the second and later calls of more than 16 steps run
    # as captured chunks; a call with events, a shorter one, a host write and a
    # longer one than the drive ring come between
    net = _net(3000, 60, delay_max=40, seed=6, inhib=0.2, w=(0.05, 0.3))

    def events(i, steps):
        m = 20 if i == 3 else 0
        return np.arange(m) % 30 + 1, np.arange(m), np.zeros(m)
    _both(net, _drive(3000, seed=6, bg=0.003), 1.0, [40, 40, 33, 40, 17, 40, 1100, 5, 40], events=events)


# where the networks lie: one alone past the first slice, two in one run of
# slices, two with a hole between them that the active list covers (small) or
# leaves out (large); weights written with spikes in flight change sign class
@pytest.mark.parametrize("keep,hole", [((2,), 300), ((1, 2), 300), ((0, 2), 100), ((0, 2), 9000)])
@pytest.mark.parametrize("n,k", [(1500, 30), (24_000, 25)])
def test_where_networks_lie(keep, hole, n, k):
    nets = [_net(n, k, seed=1), _net(hole, 10, seed=2), _net(n + 65, k, seed=3)]

    def run(sim, ids):
        out = []
        for c in range(3):
            sim.step(25)
            for j, i in ids.items():
                w = sim.weights(i, nets[j].n_syn)
                out += [w, sim.potential(i, nets[j].n), sim.firings(i, nets[j].n)]
                if c == 1:
                    sim.write_weights(i, np.where(np.arange(w.size) % 3 == 0, -w, w))
        return out + [x for j, i in ids.items() for x in _state(sim, i, nets[j])]

    sim = nc.Simulation(sum(m.n + 64 for m in nets), sum(m.n_syn for m in nets), 4)
    ids = [sim.add(m, None, _drive(m.n, j)) for j, m in enumerate(nets)]
    for j in range(3):
        if j not in keep:
            sim.remove(ids[j])
    got = run(sim, {j: ids[j] for j in keep})
    sim.close()
    want = {}
    for j in keep:
        sim = nc.Simulation.for_network(nets[j])
        sim.set_launch(**PER_SLICE)
        want[j] = run(sim, {j: sim.add(nets[j], None, _drive(nets[j].n, j))})
        sim.close()
    calls = [x for c in range(3) for j in keep for x in want[j][3 * c:3 * c + 3]]  # three arrays a call
    _same(got, calls + [x for j in keep for x in want[j][9:]])


@pytest.mark.parametrize("sync", [True, False])
def test_own_graphs_made_and_updated(sync):
    # a long first call makes the graph behind its first steps (96); networks
    # that join, stop and leave change its launches, which later calls of 48
    # steps or more give it when the device is idle, and launch directly when
    # the calls before still run
    nets = [_net(n, 40, delay_max=40, seed=n, inhib=0.2, w=(0.05, 0.3)) for n in (3000, 1500, 9000, 2000)]
    got = []
    for shape in ({}, PER_SLICE):
        sim = nc.Simulation(sum(m.n + 64 for m in nets), sum(m.n_syn for m in nets), 4)
        sim.set_launch(**shape)
        add = lambda j, steps=0: sim.add(nets[j], None, _drive(nets[j].n, j, bg=0.002), steps=steps)
        ids = {0: add(0)}
        out = []
        for steps, join, left in ((143, None, None), (144, 1, None), (200, 2, None), (48, None, 1), (47, 3, None),
                                  (1300, None, None), (60, None, 0), (60, 1, None), (15, None, None)):
            sim.step(steps)
            if left is not None:
                out += _state(sim, ids[left], nets[left])
                sim.remove(ids.pop(left))
            if join is not None:
                ids[join] = add(join, 250 if join == 2 else 0)
            if sync:
                out += [sim.potential(i, nets[j].n) for j, i in ids.items()]
        got.append(out + [x for j, i in ids.items() for x in _state(sim, i, nets[j])])
        sim.close()
    _same(*got)
