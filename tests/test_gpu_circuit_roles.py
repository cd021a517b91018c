"""Circuits with more clocks, trains, Poisson devices, lists, folds and plastic
projections than one launch of a step holds, with every lane count of the
fold, delays whose event-queue replay fits the lists' launch and longer ones,
and both delivery orders.  Rasters, states, weights and learning state against
the oracle.
"""
import numpy as np
import pytest

import edlut_amd as E
from edlut_amd import workloads
from tests.helpers import LIF_DEFAULTS, bits, np_out_csr

pytestmark = pytest.mark.gpu

N = 60


def _edges(rng, n_src, per, lo, hi, w):
    e = n_src * per
    return (np.repeat(np.arange(n_src, dtype=np.int32), per), rng.integers(0, N, e).astype(np.int32),
            rng.integers(lo, hi + 1, e).astype(np.int32), np.zeros(e, np.uint8),
            rng.uniform(0, w, e).astype(np.float32))


@pytest.mark.parametrize("hi,graph,queue", [(6, True, True), (6, False, True), (64, True, True), (65, True, True),
                                            (6, True, False)])
def test_more_roles_than_a_launch(oracle, hi, graph, queue):
    steps = 220
    print(f"case roles delays<={hi} graph={graph} queue={queue}", flush=True)
    rng = np.random.default_rng(hi)
    dt = float(np.float32(1e-4))
    models, nets, opops, onets = [], [], [], []
    for i in range(6):
        m = E.CreateNeuronModel("LIFTimeDrivenModel_GPU", {"int_meth": E.integration_method("Euler", dt)})
        m.CheckSynapseType(0)
        m.InitializeStates(N, 0, 0)
        models.append(m)
        nets.append(E.Network(m, hi))
        o = oracle.Population("LIFTimeDrivenModel_GPU", "Euler", LIF_DEFAULTS, N, dt_s=np.float32(1e-4), mask=1)
        opops.append(o)
        onets.append(oracle.Net(o, hi))
        nets[i].set_graph(graph)
        nets[i].set_event_order(queue)
        nets[i].set_launch(4, (8, 16, 32, 64, 8, 16)[i], (3, 64, 512, 17, 64, 5)[i])
    for i in range(6):   # 0-2: delivery one update ahead; 3-5: plastic
        if i < 5:
            states, ed = workloads.lcg_seeds(77 + i, 300), _edges(rng, 300, 12, 1, hi, 3.0)
            nets[i].add_poisson(states, 200.0, *E.build_out_csr(300, N, hi, *ed))
            onets[i].add_poisson(states, 200.0, *np_out_csr(300, N, hi, *ed))
        for _ in range((2, 2, 1, 0, 0, 0)[i]):
            cnt = rng.integers(0, 4, steps)
            ptr = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
            idx = np.concatenate([np.sort(rng.choice(40, c, replace=False)) for c in cnt]).astype(np.int32)
            ed = _edges(rng, 40, 10, 1, hi, 2.0)
            nets[i].add_spike_train(40, ptr, idx, *E.build_out_csr(40, N, hi, *ed))
            onets[i].add_train(40, ptr, idx, *np_out_csr(40, N, hi, *ed))
        for j in ((i + 1) % 6, (i + 2) % 6, (i + 3) % 6)[:3 if i >= 3 else 1]:
            ed = _edges(rng, N, 20, 1, hi, 1.5)
            nets[i].add_projection(nets[j], *E.build_out_csr(N, N, hi, *ed))
            onets[i].add_link(onets[j], *np_out_csr(N, N, hi, *ed))
    plastic = [(3, 1), (3, 2), (3, 3), (4, 1), (4, 2), (4, 3), (5, 0), (5, 1), (5, 2)]
    for i, s in plastic:
        nets[i].set_stdp(s, 0.02, 0.01, 0.015, 0.02, 3.0)
        onets[i].set_stdp(s, 0.02, 0.01, 0.015, 0.02, 3.0)
    circuit = E.Circuit(nets)
    if not queue:
        oracle.set_order(0)
    try:
        for k, m in ((1, 90), (91, 5), (96, steps - 95)):
            circuit.run(m)
            oracle.circuit_run(onets, k, m)
    finally:
        oracle.set_order(1)
    for i in range(6):
        st, ix = nets[i].spikes()
        ost, oix = onets[i].take_log()
        assert len(ost) > 10, f"network {i} should fire"
        assert np.array_equal(st, ost) and np.array_equal(ix, oix), f"network {i} raster"
        for v in range(opops[i].nv):
            assert np.array_equal(bits(models[i].GetVectorNeuronState(v)), bits(opops[i].state(v))), f"{i} var {v}"
    for i, s in plastic:
        w_o, pre_o, post_o, last_o = onets[i].synapses(s)
        _, _, w_g = nets[i].synapses(s)
        pre_g, post_g, last_g = nets[i].stdp_state(s)
        assert np.array_equal(bits(w_g), bits(w_o)), f"weights {i}/{s}"
        assert np.array_equal(bits(pre_g), bits(pre_o)) and np.array_equal(bits(post_g), bits(post_o))
        assert np.array_equal(last_g.view(np.uint64), last_o.view(np.uint64))
    circuit.close()
