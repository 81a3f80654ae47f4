"""A simulation that takes much of the device's memory has arrival buckets of 64
entries instead of 128: its networks go through the same states, in every form
of the step kernels.  (Room for 2e9 synapses takes about 95 GB, most of which is
never touched.)"""
import numpy as np
import pytest

import neurocorrelation_amd as nc
from neurocorrelation_amd import workloads as W

pytestmark = pytest.mark.gpu

LARGE = dict(max_synapses=2_000_000_000, max_slots=2_600_000_000)


def _sim(nets, large):
    pos = sum(m.device_size()[0] for m in nets)
    if large:
        return nc.Simulation(pos, max_nets=len(nets), raster_capacity=1 << 18, **LARGE)
    return nc.Simulation(pos, sum(m.n_syn for m in nets), len(nets), 1 << 18,
                         max_slots=sum(m.device_size()[1] for m in nets))


def _burst():
    """320 spikes into one slice at one step."""
    src = np.arange(64, 64 + 320)
    return src, nc.Network.from_edges(400, np.repeat(np.arange(8), 40), src, np.full(320, 0.4, np.float32),
                                      np.full(320, 9, np.uint8))


@pytest.mark.parametrize("large,room", [(False, 128), (True, 64)])
def test_room_of_a_bucket(large, room):
    src, net = _burst()
    sim = _sim([net], large)
    i = sim.add(net)
    sim.set_counting(True)  # the counters are the per-slice kernels'
    sim.push_forced(i, np.ones(320), src, np.zeros(320))
    sim.step(10)
    assert sim.counters()["bucket_entries"] == room
    sim.close()


# a workgroup per network, several waves per slice, a wave per slice (in-degrees
# past the others'), an explicit shape: networks in which 64 to 128 and more
# spikes arrive at a slice in a step
@pytest.mark.parametrize("n,k,shape", [(400, 0, {}), (900, 50, {}), (3000, 50, {}), (2000, 300, {}),
                                       (3000, 50, dict(waves_per_block=2)), (1500, 50, dict(persistent=1))])
def test_states_are_the_same(n, k, shape):
    src, net = _burst()
    if k:
        net = nc.Network.generate(n, W.side_for(n), W.radius_for_degree(k), 1, 20, 0.2, 0.8, seed=n)
    drive = None if not k else W.drive_spec(dict(n_inputs=n // 20, n_groups=2, n_correlated=2, period=200, p0=0.05,
                                                 amp_corr=1.0, amp_ind=0.5), seed=1)
    states = []
    for large in (False, True):
        sim = _sim([net], large)
        i = sim.add(net, None, drive)
        sim.set_launch(**shape)
        out = []
        for steps in (12, 40, 40):
            if not k:
                sim.push_forced(i, np.ones(320), src, np.zeros(320))
            sim.step(steps)
            out += [sim.save(i), *sim.raster(i, 1 << 18)]
        states.append(out)
        sim.close()
    assert all(np.array_equal(a, b) for a, b in zip(*states))
