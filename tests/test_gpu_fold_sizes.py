"""Events per key and step from none to 40: single events, the four sorted in
registers, and the passes over more of them (their eight-entry blocks and
four-event passes just full and just over), in several keys of one lane at
once, with the event queue's order and the canonical one.  Poisson devices
that fire at every step give a target as many events per step as it has
synapses; magnitudes differ so that any other order of addition changes the
bits.  State and raster against the oracle.
"""
import numpy as np
import pytest

import edlut_amd as E
from edlut_amd import workloads
from tests.helpers import bits, defaults, np_out_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("queue", [True, False])
@pytest.mark.parametrize("model,integ,n", [("LIFTimeDrivenModel_GPU", "Euler", 1100),
                                           ("AdExTimeDrivenModel_GPU", "RK4", 1100),
                                           ("HHTimeDrivenModel_GPU", "BDF", 600),
                                           ("EgidioGranuleCell_TimeDriven_GPU", "BDF", 90)])
def test_events_per_key(oracle, model, integ, n, queue):
    print(f"case events per key {model} queue={queue}", flush=True)
    hi, steps, n_src = 5, 24, 64
    rng = np.random.default_rng(n)
    exc = np.array([0, 1, 2, 3, 4, 5, 7, 8, 9, 12, 13, 16, 17, 40])[np.arange(n) % 14]
    inh = np.array([0, 1, 2, 4, 6, 0, 0, 3, 1, 0, 10])[np.arange(n) % 11]
    tgt = np.concatenate([np.repeat(np.arange(n), exc), np.repeat(np.arange(n), inh)]).astype(np.int32)
    typ = np.concatenate([np.zeros(exc.sum(), np.uint8), np.ones(inh.sum(), np.uint8)])
    src = rng.integers(0, n_src, len(tgt)).astype(np.int32)
    delay = rng.integers(1, hi + 1, len(tgt)).astype(np.int32)
    w = (10.0 ** rng.uniform(-6, -1, len(tgt))).astype(np.float32)
    m = E.CreateNeuronModel(model, {"int_meth": E.integration_method(integ, 1e-4, 2)})
    for t in (0, 1):
        m.CheckSynapseType(t)
    m.InitializeStates(n, 0, 0)
    o = oracle.Population(model, integ, defaults(model), n, dt_s=np.float32(1e-4), mask=3, bdf_order=2)
    net, onet = E.Network(m, hi), oracle.Net(o, hi)
    net.set_event_order(queue)
    for half in (src < 20, src >= 20):   # two devices
        states = workloads.lcg_seeds(5 + int(half[0]), n_src)
        ed = (src[half], tgt[half], delay[half], typ[half], w[half])
        net.add_poisson(states, 2e4, *E.build_out_csr(n_src, n, hi, *ed))
        onet.add_poisson(states, 2e4, *np_out_csr(n_src, n, hi, *ed))
    if not queue:
        oracle.set_order(0)
    try:
        for k, c in ((1, 17), (18, steps - 17)):
            net.run(c)
            ost, oix = onet.run(k, c)
    finally:
        oracle.set_order(1)
    for v in range(o.nv):
        assert np.array_equal(bits(m.GetVectorNeuronState(v)), bits(o.state(v))), f"variable {v}"
    st, ix = net.spikes()
    late = st >= 18
    assert np.array_equal(st[late], ost) and np.array_equal(ix[late], oix)
