"""Pulled delivery of grouped populations (dense groups read their incoming
lists, quiet ones push their events): every group equals the same network run
alone as a plain population, whichever way its events take, while groups
change over, over runs of any split, for arbitrary synapse lists, and where
the lists cannot be pulled.
"""
import numpy as np
import pytest

import edlut_amd as E
from edlut_amd.network import Network, binomial_thresholds, build_out_csr
from tests.helpers import ADEX_DEFAULTS, bits

pytestmark = pytest.mark.gpu
MODEL = "AdExTimeDrivenModel_GPU"
THR = binomial_thresholds(100, 5.0 * 1e-4)


def _group(sizes, params, max_d):
    m = E.CreateNeuronModel(MODEL, {"int_meth": E.integration_method("RK4", 1e-4)})
    m.InitializeGroups(np.asarray(sizes, np.int32), params)
    return m, Network(m, max_d)


def _alone(n, params, max_d):
    names = [k for k, _ in E.REGISTRY[MODEL].PARAMS]
    m = E.CreateNeuronModel(MODEL, {k: float(v) for k, v in zip(names, params)})
    m.SetParameters({"int_meth": E.integration_method("RK4", 1e-4)})
    m.InitializeStates(int(n))
    net = Network(m, max_d)
    net.set_event_order(False)
    return m, net


def _equal(gm, gnet, g, pm, pnet, n):
    start, _ = gm.GetGroups()
    gst, gix = gnet.spikes()
    sel = (gix >= start[g]) & (gix < start[g] + n)
    pst, pix = pnet.spikes()
    assert np.array_equal(gst[sel], pst) and np.array_equal(gix[sel] - start[g], pix), f"group {g}: raster"
    for v in range(4):
        a = gm.GetVectorNeuronState(v)[start[g]:start[g] + n]
        assert np.array_equal(bits(a), bits(pm.GetVectorNeuronState(v))), f"group {g} variable {v}"
    return len(pst) / (n * max(gnet.next_step - 1, 1))


@pytest.mark.parametrize("graph,items", [(True, 4), (False, 2)])
def test_mixed_groups(graph, items):
    """Rates from silence to saturation, rising through the run."""
    sizes = [33, 256, 1000, 4100, 257, 9000]
    params = np.tile(ADEX_DEFAULTS, (len(sizes), 1))
    params[:, 8] = [-65.0, -75.0, -55.0, -50.0, -95.0, -54.0]
    max_d, runs = 7, (1, 5, 16, 37, 150, 16, 90)
    print(f"case mixed groups graph={graph} items={items}", flush=True)
    gm, gnet = _group(sizes, params, max_d)
    gnet.generate_recurrent(80, 0.8, -0.5, 0.5, 99)
    gnet.set_external(THR, 2.0, 7)
    gnet.set_launch(items, 32, 256)
    gnet.set_graph(graph)
    for _ in range(2):     # the second time after a reset
        for r in runs:
            gnet.run(r)
        rates = []
        for g, n in enumerate(sizes):
            pm, pnet = _alone(n, params[g], max_d)
            pnet.generate_recurrent(80, 0.8, -0.5, 0.5, 99 + g)
            pnet.set_external(THR, 2.0, 7 + g)
            for r in runs:
                pnet.run(r)
            rates.append(_equal(gm, gnet, g, pm, pnet, n))
            pnet.close()
            pm.close()
        assert max(rates) > 0.02 and min(rates) < 0.002, rates
        assert 0 < gnet.pulled_groups() < len(sizes)
        gnet.reset()


def _random_edges(rng, n, e, max_d, hub):
    # duplicates of one (source, target, delay), targets without synapses, a hub
    src = rng.integers(0, n, e).astype(np.int32)
    tgt = rng.integers(0, max(1, n * 7 // 8), e).astype(np.int32)
    tgt[: min(hub, e)] = 0
    src[e // 2: e // 2 + e // 8] = src[: e // 8]
    tgt[e // 2: e // 2 + e // 8] = tgt[: e // 8]
    delay = rng.integers(1, max_d + 1, e).astype(np.int32)
    delay[e // 2: e // 2 + e // 8] = delay[: e // 8]
    return src, tgt, delay, (rng.random(e) < 0.3).astype(np.uint8), rng.lognormal(1.0, 1.0, e).astype(np.float32)


@pytest.mark.parametrize("lists,hub,between", [(True, 100, False), (False, 100, True), (False, 3000, False)])
def test_given_synapses(lists, hub, between):
    """Incoming lists of every length, none and one synapse among them; some
    synapses between groups, or a hub with more synapses than a list can take,
    keep delivery with the push fold."""
    sizes, max_d = [300, 1500, 1], 5
    print(f"case given synapses lists={lists} hub={hub} between={between}", flush=True)
    params = np.tile(ADEX_DEFAULTS, (3, 1))
    gm, gnet = _group(sizes, params, max_d)
    start, _ = gm.GetGroups()
    rng = np.random.default_rng(4)
    edges = [_random_edges(rng, n, 40 * n, max_d, hub) for n in sizes]
    src = np.concatenate([e[0] + s for e, s in zip(edges, start)])
    tgt = np.concatenate([e[1] + s for e, s in zip(edges, start)])
    rest = [np.concatenate([e[j] for e in edges]) for j in (2, 3, 4)]
    if between:
        src[::97] = (src[::97] + 256) % 300
    csr = build_out_csr(gm.size, gm.size, max_d, src, tgt, *rest)
    gnet.add_recurrent(*csr)
    pm, pnet = _alone(gm.size, ADEX_DEFAULTS, max_d)
    pnet.add_recurrent(*csr)
    v = np.full(gm.size, -65.0, np.float32)
    for s, n in zip(start, sizes):
        v[s:s + n] = rng.uniform(-60, -20, n)
    gm.SetVectorNeuronState(0, v)
    pm.SetVectorNeuronState(0, v)
    pulled = []
    for r in (3, 40, 80):
        gnet.run(r)
        pnet.run(r)
        pulled.append(gnet.pulled_groups())
    assert max(pulled) > 0 if lists else set(pulled) == {-1}, pulled
    a, b = gnet.spikes(), pnet.spikes()
    assert len(a[0]) > 0.01 * 123 * gm.size
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    for s, n in zip(start, sizes):
        for k in range(4):
            assert np.array_equal(bits(gm.GetVectorNeuronState(k)[s:s + n]),
                                  bits(pm.GetVectorNeuronState(k)[s:s + n])), f"variable {k}"


def test_source_added_between_runs():
    """A Poisson source added while dense groups are pulled: their events come
    through the push fold from then on, none lost or delivered twice."""
    sizes, max_d = [500, 900], 6
    print("case source added", flush=True)
    params = np.tile(ADEX_DEFAULTS, (2, 1))
    params[:, 8] = -50.0
    gm, gnet = _group(sizes, params, max_d)
    gnet.generate_recurrent(80, 0.8, -0.5, 0.5, 5)
    gnet.set_external(THR, 2.0, 3)
    alone = []
    for g, n in enumerate(sizes):
        pm, pnet = _alone(n, params[g], max_d)
        pnet.generate_recurrent(80, 0.8, -0.5, 0.5, 5 + g)
        pnet.set_external(THR, 2.0, 3 + g)
        alone.append((pm, pnet))
    nets = [gnet] + [p[1] for p in alone]
    for net in nets:
        net.run(150)
        assert net is not gnet or net.pulled_groups() == len(sizes)
        empty = np.zeros(0, np.int32)
        net.add_poisson(np.arange(1, 4, dtype=np.uint32), 0.0,
                        *build_out_csr(3, net.model.size, max_d, empty, empty, empty, empty.astype(np.uint8),
                                       empty.astype(np.float32)))
        net.run(100)
        assert net.pulled_groups() == -1
    for g, n in enumerate(sizes):
        assert _equal(gm, gnet, g, *alone[g], n) > 0.02
