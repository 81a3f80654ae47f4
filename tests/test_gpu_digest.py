"""The digest of a served job's result, computed on the device, against
nc_digest (FNV-1a, pinned to published vectors in test_serve_wire.py) of the
same job's arrays read from a run alone: sizes on either side of where the
device takes it up, of a segment (256 words) and of a group of 64."""
import pytest

from neurocorrelation_amd import serve, workloads as W

pytestmark = pytest.mark.gpu


# words: 2 n + n_syn; n of 30..32 synapses per neuron
@pytest.mark.parametrize("n,k", [(300, 20), (420, 60), (520, 60), (1030, 35), (2050, 40), (3000, 90), (9000, 12)])
def test_served_digest_equals_the_host_digest(n, k):
    spec = dict(wiring=dict(n_neurons=n, side=W.side_for(n), radius=W.radius_for_degree(k), delay_min=1, delay_max=32,
                            w_min=0.05, w_max=0.3, inhib_frac=0.2, seed=n),
                drive=dict(n_inputs=n // 20, n_groups=4, n_correlated=4, period=200, p0=0.05, amp_corr=1.0,
                           amp_ind=1.0, seed=n), steps=60)
    server = serve.Server(max_neurons=20_000, max_synapses=2_000_000, max_nets=4, lanes=1)
    server.submit(1, spec)
    got = []
    while not got:
        got = server.poll(wait=10.0)
    server.close()
    want, _ = serve.run_alone(spec)
    assert got[0]["status"] == "ok"
    assert got[0]["digest"] == want["digest"] and got[0]["spikes"] == want["spikes"]
