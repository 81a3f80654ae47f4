"""What the default launch shape chooses, by nc_sim_last_launch, and that any
other shape is launched as it was given."""
import numpy as np
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


def test_the_tuner_times_the_default_shape_as_repeated_calls_run():
    # no capture in the timed trial (the last launch that the tuner made), a
    # chunk captured before it, also with another shape's graph at hand
    sim, _ = _quiet(3000)
    for before in ((), (dict(waves_per_block=4, graph_steps=16),)):
        for steps in (40, 100):
            sim.tune_list(list(before) + [{}], steps_per_trial=steps, rounds=1)
            info = sim.last_launch()
            assert (info["graph_steps"], info["graph_made"], info["waves_per_slice"]) == (16, 0, 4)
    sim.close()


def test_the_tuner_times_the_form_of_the_activity_it_has():
    # busy networks of more than 1024 slices: two waves per slice once a report
    # is read, which no call before the tuner does
    n, count = 1500, 48
    nets = [nc.Network.generate(n, W.side_for(n), W.radius_for_degree(25), 1, 20, 0.2, 0.8, seed=i, device=0)
            for i in range(count)]
    drive = W.drive_spec(dict(n_inputs=75, n_groups=2, n_correlated=2, period=200, p0=0.05, amp_corr=1.0,
                              amp_ind=0.5), seed=1)
    sim = nc.Simulation(count * (n + 64), sum(m.n_syn for m in nets), count)
    for m in nets:
        sim.add(m, None, drive)
    sim.step(80)
    assert sim.last_launch()["waves_per_slice"] == 0
    sim.tune_list([dict(waves_per_block=2), {}], steps_per_trial=16, rounds=1)
    assert sim.last_launch()["waves_per_slice"] == 2
    sim.close()


# networks of a slice (the device holds 512 of their workgroups), of a slice
# with one of 16 among them (256), of 5 slices: a round, a few, many
@pytest.mark.parametrize("count,n,one,forms", [(500, 64, 0, (1, 1, 1)), (6000, 64, 0, (0, 0, 0)),
                                               (2500, 64, 1000, (0, 0, 0)), (300, 300, 0, (1, 0, 1))])
def test_many_small_networks(count, n, one, forms):
    # a workgroup per network while the rounds they follow one another in are
    # few; whatever is chosen, a network's state is that of an explicit shape
    made = [nc.Network.generate(m, W.side_for(m), W.radius_for_degree(20), 1, 20, 0.05, 0.3, 0.2, seed=m + i)
            for i in range(4) for m in (n, one) if m]
    drive = W.drive_spec(dict(n_inputs=6, n_groups=2, n_correlated=2, period=200, p0=0.05, amp_corr=1.0,
                              amp_ind=1.0), seed=1)
    nets = [made[i % len(made)] if not one or i == 7 else made[2 * (i % 4)] for i in range(count)]
    if one:
        nets[7] = made[1]
    states = []
    for shape in ({}, dict(waves_per_block=2)):
        sim = nc.Simulation(sum(m.n + 64 for m in nets), sum(m.n_syn for m in nets), count,
                            max_slots=sum(m.device_size()[1] for m in nets))
        ids = [sim.add(m, None, drive) for m in nets]
        sim.set_launch(**shape)
        out = []
        for steps, form in zip((50, 1, 50), forms):
            sim.step(steps)
            assert sim.last_launch()["networks"] == (0 if shape else form), steps
            out += [sim.save(ids[i]) for i in (0, 7, count // 2, count - 1)]
        out += [sim.firings(i, m.n) for i, m in zip(ids, nets)]
        states.append(out)
        sim.close()
    assert all(np.array_equal(a, b) for a, b in zip(*states))
