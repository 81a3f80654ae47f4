"""What the default launch shape chooses, by nc_sim_last_launch, and that any
other shape is launched as it was given."""
import pytest

import neurocorrelation_amd as nc
from neurocorrelation_amd import workloads as W

pytestmark = pytest.mark.gpu


def _quiet(n, count=1):
    nets = [nc.Network.generate(n, W.side_for(n), W.radius_for_degree(20), 1, 20, 0.05, 0.3, 0.2, seed=1 + i % 8)
            for i in range(count)]
    sim = nc.Simulation(sum(m.device_size()[0] for m in nets), sum(m.n_syn for m in nets), count,
                        max_slots=sum(m.device_size()[1] for m in nets))
    drive = W.drive_spec(dict(n_inputs=n // 20, n_groups=2, n_correlated=2, period=200, p0=0.05, amp_corr=1.0,
                              amp_ind=1.0), seed=1)
    return sim, [sim.add(m, None, drive) for m in nets]


OTHERS = [dict(waves_per_block=2), dict(waves_per_block=8), dict(waves_per_block=4, xcd_swizzle=1),
          dict(waves_per_block=4, stage_tables=1), dict(waves_per_block=4, fanout_waves=1024),
          dict(waves_per_block=4, persistent=1)]


@pytest.mark.parametrize("shape", OTHERS)
def test_a_shape_without_graphs_launches_directly(shape):
    # equal calls, and one long enough that the default shape captures behind
    # its first steps
    sim, _ = _quiet(3000)
    sim.set_launch(**shape)
    for steps in (40, 40, 40, 300):
        sim.step(steps)
        sim.synchronize()
        assert sim.last_launch() == dict(networks=0, waves_per_slice=0, graph_steps=0, graph_made=0)
    sim.close()


def test_the_default_shape_captures_its_own():
    sim, _ = _quiet(3000)
    made = []
    for steps in (40, 40, 40, 10, 40):
        sim.step(steps)
        sim.synchronize()
        info = sim.last_launch()
        assert info["networks"] == 0 and info["waves_per_slice"] == 4
        made.append((info["graph_steps"], info["graph_made"]))
    assert made == [(0, 0), (16, 1), (16, 0), (0, 0), (16, 0)]
    # the caller's own chunks
    sim.set_launch(graph_steps=8)
    sim.step(24)
    assert sim.last_launch() == dict(networks=0, waves_per_slice=0, graph_steps=8, graph_made=1)
    sim.close()
    sim, _ = _quiet(300)
    sim.step(40)
    assert sim.last_launch() == dict(networks=1, waves_per_slice=0, graph_steps=0, graph_made=0)
    sim.close()
