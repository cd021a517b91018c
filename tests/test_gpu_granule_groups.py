"""Granule BDF kernel: a neuron on 16 lanes, bit for bit against the oracle at
the sizes where its launch changes (a wave's last group empty, four, eight and
sixteen waves per workgroup), for every order's history, and through the
reference arrangement of a Newton step with an infinite iterate.
"""
import os

import numpy as np
import pytest

import edlut_amd as E
from tests.helpers import bits, defaults

pytestmark = pytest.mark.gpu
GR = "EgidioGranuleCell_TimeDriven_GPU"


def _run(oracle, n, order, steps, infinite=()):
    print(f"case granule groups n={n} order={order} steps={steps}", flush=True)
    rng = np.random.default_rng(n + 1000 * order)
    m = E.CreateNeuronModel(GR, {"int_meth": E.integration_method("BDF", 1e-4, order)})
    for t in (0, 1, 2):
        assert m.CheckSynapseType(t)
    m.InitializeStates(n, 0, 0)
    o = oracle.Population(GR, "BDF", defaults(GR), n, dt_s=np.float32(1e-4), mask=15, bdf_order=order)
    cur = rng.uniform(0.0, 200.0, n).astype(np.float32)
    m.ProcessInputCurrent(cur)
    o.set_ext_current(cur)
    oracle.set_threads(min(16, os.cpu_count() or 1))
    total = 0
    try:
        for k in range(1, steps + 1):
            if k == 6:
                for var, i in infinite:
                    v = m.GetVectorNeuronState(var)
                    v[i] = np.inf
                    m.SetVectorNeuronState(var, v)
                    ov = o.state(var)
                    ov[i] = np.inf
                    o.set_state(var, ov)
            ne = max(1, n // 4)
            tgt = rng.integers(0, n, ne).astype(np.int32)
            typ = rng.choice(np.array([0, 0, 0, 1, 2], np.uint8), ne)
            w = rng.uniform(0.0, 1.0, ne).astype(np.float32)
            m.ProcessInputSpikes(tgt, typ, w)
            o.add_inputs(tgt, typ, w)
            m.UpdateState(step=k)
            ref = o.update(k)
            assert np.array_equal(m.GetInternalSpikeIndexs(), ref), f"update {k}"
            total += len(ref)
    finally:
        oracle.set_threads(1)
    for v in range(o.nv):
        assert np.array_equal(bits(m.GetVectorNeuronState(v)), bits(o.state(v))), f"var {v}"
    return total


@pytest.mark.parametrize("n,order,steps", [(5, 3, 200), (63, 6, 200), (31, 4, 100), (1023, 1, 60), (4096, 2, 60),
                                           (4097, 2, 60), (32_769, 2, 50)])
def test_group_shapes(oracle, n, order, steps):
    assert _run(oracle, n, order, steps) > 0


def test_infinite_iterate(oracle):
    """An infinite V, gate or calcium concentration is no NaN yet: the Newton
    step takes the reference's arrangement and makes it one."""
    _run(oracle, 70, 2, 40, infinite=[(0, 2), (0, 66), (1, 5), (10, 21), (11, 33), (14, 69)])
