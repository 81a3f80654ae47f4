"""Wiring on the GPU against the host builder, bit for bit, at the edges of the
device builder's work split: items of up to 64 targets of a cell, candidates in
LDS up to 2048 at a time (past that in pieces in Morton order, and by the sort
of all pairs in draw order), cells with no or one member."""
import numpy as np
import pytest

import neurocorrelation_amd as nc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spatial", [0, 1])
@pytest.mark.parametrize("n,side,radius", [
    (1, 1.0, 0.5),          # nothing to wire
    (2, 1.0, 5.0),          # one cell, both in it
    (64, 1.0, 2.0),         # one full item
    (65, 1.0, 2.0),         # an item of one target
    (129, 1.0, 0.9),        # one cell per axis, part of it in reach
    (2048, 1.0, 0.3),       # one cell's candidates fill the LDS list exactly in reach of 27 cells
    (2049, 1.0, 0.6),       # one past it
    (5000, 1.0, 0.55),      # one cell of 5000: three pieces
    (6000, 1.0, 0.34),      # two cells per axis, every cell sees all 6000
    (700, 40.0, 1.0),       # mostly empty cells
    (20_000, 4.0, 0.431),   # the dense workload's scale, ragged
    (33_333, 20.0, 0.2)])   # 100 cells per axis, 0.03 a cell
def test_device_rows_equal_the_host_builder(n, side, radius, spatial):
    args = dict(n_neurons=n, side=side, radius=radius, delay_min=2, delay_max=200, w_min=0.1, w_max=0.7,
                inhib_frac=0.3, seed=n + spatial, spatial_order=spatial)
    host, dev = nc.Network.generate(**args), nc.Network.generate(device=0, **args)
    assert host.info() == dev.info()
    a, b = host.export(), dev.export()
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), k
