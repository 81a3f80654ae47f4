"""nc_read_weights_noalloc beyond what goes through the simulation's own pinned
buffer: no thread is started (each takes a thread id, which the kernel counts
up) and no host memory is mapped, in a process whose first large read it is;
the weights equal the allocating read's."""
import threading

import numpy as np
import pytest

import neurocorrelation_amd as nc
from neurocorrelation_amd import workloads as W

pytestmark = pytest.mark.gpu


def _new_thread_id():
    t = threading.Thread(target=lambda: None)
    t.start()
    t.join()
    return t.native_id


def _mapped_kib():
    for line in open("/proc/self/status"):
        if line.startswith("VmSize:"):
            return int(line.split()[1])


# 1 MiB of weights is the pinned buffer's; from 2 MiB on, reads that may
# allocate take several threads
@pytest.mark.parametrize("n,k", [(3000, 60), (40_000, 60)])
def test_large_read_starts_no_thread(n, k):
    net = nc.Network.generate(n, W.side_for(n), W.radius_for_degree(k), 1, 20, seed=3)
    assert (4 * net.n_syn > 2 << 20) == (n > 3000)
    sim = nc.Simulation.for_network(net)
    i = sim.add(net)
    out = np.zeros(net.n_syn, np.float32)
    read = lambda: nc.engine.check(nc.lib().nc_read_weights_noalloc(
        sim._h, i, out.ctypes.data_as(nc._lib.C.POINTER(nc._lib.C.c_float)), net.n_syn))
    read()
    ids, grown = [], []
    for _ in range(20):
        a, m0 = _new_thread_id(), _mapped_kib()
        read()
        grown.append(_mapped_kib() - m0)
        ids.append(_new_thread_id() - a)
    # other processes may take ids meanwhile, but not in each of the calls
    assert min(x for x in ids if x > 0) == 1, ids
    assert min(grown) == 0, grown
    assert np.array_equal(out, sim.weights(i, net.n_syn))
    sim.close()
