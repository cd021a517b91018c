"""The replayed event queue at every depth of its heap: heaps inside one
six-level block, across two blocks in 16 KB and in 64 KB of LDS, and larger
ones that stay in memory across three blocks.  Raster, state and the stored
heap, entry by entry, against the oracle.
"""
import numpy as np
import pytest

import edlut_amd as E
from edlut_amd import workloads
from tests.helpers import LIF_DEFAULTS, bits, np_out_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("lo,hi,steps", [(1, 1, 80), (1, 6, 100), (1, 12, 150), (5, 40, 200), (10, 64, 300),
                                         (20, 90, 320), (30, 120, 420)])
def test_heap_depths(oracle, lo, hi, steps, graph):
    print(f"case heap depths delays {lo}-{hi} graph={graph}", flush=True)
    n, per = 40, 30
    rng = np.random.default_rng(hi)
    states = workloads.lcg_seeds(1000 + hi, n * per)
    e = n * per
    poisson = (np.arange(e, dtype=np.int32), np.repeat(np.arange(n, dtype=np.int32), per),
               rng.integers(lo, hi + 1, e).astype(np.int32), (np.arange(e) % 5 == 0).astype(np.uint8),
               rng.uniform(0, 1.5, e).astype(np.float32))
    r = n * 20
    rec = (rng.integers(0, n, r).astype(np.int32), rng.integers(0, n, r).astype(np.int32),
           rng.integers(lo, hi + 1, r).astype(np.int32), np.zeros(r, np.uint8),
           rng.uniform(0, 0.3, r).astype(np.float32))
    spec = workloads.NetworkSpec("LIFTimeDrivenModel_GPU", "Euler", n, hi, rec=rec, steps=steps)
    spec.poisson.append((states, 60.0, poisson))
    model, net = E.from_spec(spec)
    net.set_graph(graph)
    pop, onet = oracle.from_spec(spec, LIF_DEFAULTS, np_out_csr)
    ost, oix = [], []
    for k, m in ((1, steps // 2), (1 + steps // 2, steps - steps // 2)):
        net.run(m)
        a, b = onet.run(k, m)
        ost.append(a)
        oix.append(b)
        t_d, key_d = net.event_queue()
        t_o, prio, kind, _, d = onet.event_queue()
        assert len(t_d) == len(t_o)
        assert np.array_equal(t_d.view(np.uint64), t_o.view(np.uint64))
        # priority, kind and delay (the two sides number the models themselves)
        key_o = (prio.astype(np.uint32) << 28) | (kind.astype(np.uint32) << 24) | d.astype(np.uint32)
        assert np.array_equal(key_d & np.uint32(0xff00ffff), key_o)
    st, ix = net.spikes()
    ost, oix = np.concatenate(ost), np.concatenate(oix)
    assert len(ost) > 10
    assert np.array_equal(st, ost) and np.array_equal(ix, oix)
    for v in range(pop.nv):
        assert np.array_equal(bits(model.GetVectorNeuronState(v)), bits(pop.state(v))), f"variable {v}"


@pytest.mark.parametrize("rate", [60.0, 1500.0, 2e4])
def test_spikes_per_wave(oracle, rate):
    """Devices of 700 sources with one synapse each (no source has every
    delay): at most a few spikes in a wave's tiles, some in every tile, and
    all 700, more than a wave's list holds."""
    print(f"case spikes per wave rate={rate}", flush=True)
    n, n_src, hi, steps = 50, 700, 9, 60
    rng = np.random.default_rng(int(rate))
    poisson = (np.arange(n_src, dtype=np.int32), rng.integers(0, n, n_src).astype(np.int32),
               rng.integers(1, hi + 1, n_src).astype(np.int32), np.zeros(n_src, np.uint8),
               (10.0 ** rng.uniform(-4, -1, n_src)).astype(np.float32))
    spec = workloads.NetworkSpec("LIFTimeDrivenModel_GPU", "Euler", n, hi, rec=None, steps=steps)
    spec.poisson.append((workloads.lcg_seeds(31, n_src), rate, poisson))
    model, net = E.from_spec(spec)
    pop, onet = oracle.from_spec(spec, LIF_DEFAULTS, np_out_csr)
    for k, m in ((1, 37), (38, steps - 37)):
        net.run(m)
        onet.run(k, m)
        t_d, _ = net.event_queue()
        t_o = onet.event_queue()[0]
        assert np.array_equal(t_d.view(np.uint64), t_o.view(np.uint64))
    for v in range(pop.nv):
        assert np.array_equal(bits(model.GetVectorNeuronState(v)), bits(pop.state(v))), f"variable {v}"
