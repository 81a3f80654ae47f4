"""Simulation.save fills a bytes object in place without touching what
ctypes.pythonapi's users share."""
import ctypes as C

import neurocorrelation_amd as nc
from neurocorrelation_amd import engine


class _Lib:
    def nc_sim_save(self, h, net_id, buf, cap, size):
        C.cast(size, C.POINTER(C.c_uint64))[0] = 100
        if buf is not None:
            assert cap == 100
            C.memmove(buf, bytes(range(100)), 100)
        return 0


def test_save_leaves_the_shared_prototypes(monkeypatch):
    shared = C.pythonapi.PyBytes_FromStringAndSize
    before = shared.restype, shared.argtypes
    monkeypatch.setattr(engine, "lib", _Lib)
    sim = nc.Simulation.__new__(nc.Simulation)
    sim._h = None
    assert sim.save(0) == bytes(range(100))
    assert sim.save(0) == bytes(range(100))
    assert (shared.restype, shared.argtypes) == before
    assert C.pythonapi.PyBytes_FromStringAndSize is shared
