"""Host-scheduled events in bulk, in no order, over networks of one simulation
that stop at their own step counts: each network's fires and state equal those
of the network alone under an explicit launch shape, whose kernels take the
events through the forced-fire bits."""
import numpy as np
import pytest

import neurocorrelation_amd as nc
from neurocorrelation_amd import workloads as W

pytestmark = pytest.mark.gpu


def _nets(sizes):
    return [nc.Network.generate(n, W.side_for(n), W.radius_for_degree(12), 1, 20, 0.05, 0.3, 0.2, seed=n)
            for n in sizes]


def _events(call, j, n, steps, per):
    """`per` events a step and network on average, some past the call."""
    rng = np.random.default_rng([call, j])
    m = per * steps if j % 3 else 0  # every third network has none
    return rng.integers(1, steps + 4, m), rng.integers(0, n, m), rng.integers(0, 2, m)


def _run(nets, of, shape, calls, per, budget):
    sim = nc.Simulation(sum(m.device_size()[0] for m in nets), sum(m.n_syn for m in nets), len(nets),
                        raster_capacity=1 << 21, max_slots=sum(m.device_size()[1] for m in nets))
    sim.set_launch(**shape)
    ids = [sim.add(m, nc.default_params(dt=0.5), steps=budget(j)) for j, m in zip(of, nets)]
    out = {j: [] for j in of}
    for c, steps in enumerate(calls):
        for j, i, m in zip(of, ids, nets):
            sim.push_forced(i, *_events(c, j, m.n, steps, per))
        sim.step(steps)
        for j, i, m in zip(of, ids, nets):
            out[j] += [sim.save(i), sim.firings(i, m.n), *sim.raster(i, 1 << 21)]
    sim.close()
    return out


# networks of a workgroup each, of several waves per slice, and of a wave per
# slice; fewer events than go through pinned memory at a time (4096), and more;
# calls of one step, of a few, and past the drive ring's 1024
@pytest.mark.parametrize("sizes", [(300, 64, 65, 700, 1, 900), (1500, 200, 2000), (20_000, 30_000, 20_000)])
@pytest.mark.parametrize("per", [2, 70])
def test_events_in_bulk(sizes, per):
    nets = _nets(sizes)
    calls = [1, 30, 1100] if sizes[0] == 300 else [1, 30]
    if per == 70 and sizes[0] == 300:
        calls = [1, 30, 1030]
    budget = lambda j: 25 if j == 2 else 0
    got = _run(nets, range(len(nets)), {}, calls, per, budget)
    for j, m in enumerate(nets):
        want = _run([m], [j], dict(waves_per_block=2), calls, per, budget)
        for a, b in zip(got[j], want[j]):
            assert np.array_equal(a, b), j
