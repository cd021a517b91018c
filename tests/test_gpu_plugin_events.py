"""Plug-in updates at the edges of their event lists and spike hand-back,
against the oracle: keys with one to many events in every order of arrival,
several pushes per update, a queue that grows, updates with more spikes than
the compaction hands back by itself, and BDF tiles that end inside a
workgroup.
"""
import numpy as np
import pytest

import edlut_amd as E
from tests.helpers import bits, defaults

pytestmark = pytest.mark.gpu
LIF, ADEX, HH = "LIFTimeDrivenModel_GPU", "AdExTimeDrivenModel_GPU", "HHTimeDrivenModel_GPU"


def _pair(oracle, model, integ, n, order=1, fp64=False):
    m = E.CreateNeuronModel(model, {"int_meth": E.integration_method(integ, 1e-4, order)})
    for t in (0, 1, 2):
        assert m.CheckSynapseType(t)
    m.InitializeStates(n, 0, 0)
    if fp64:
        m.SetNewtonFP64(True)
    o = oracle.Population(model, integ, defaults(model), n, dt_s=np.float32(1e-4), mask=7, bdf_order=order,
                          fp64=2 if fp64 else False)
    return m, o


def _step(m, o, k, tgt, typ, w, pushes=1):
    for part in np.array_split(np.arange(len(tgt)), pushes):
        m.ProcessInputSpikes(tgt[part], typ[part], w[part])
    o.add_inputs(tgt, typ, w)
    m.UpdateState(step=k)
    ref = o.update(k)
    assert np.array_equal(m.GetInternalSpikeIndexs(), ref), f"update {k}"
    return len(ref)


def _state(m, o):
    for v in range(o.nv):
        assert np.array_equal(bits(m.GetVectorNeuronState(v)), bits(o.state(v).astype(np.float32))), f"var {v}"


@pytest.mark.parametrize("per_key", [1, 2, 3, 4, 5, 8, 9, 33, 96, 97, 200, 5000])
def test_events_of_one_key(oracle, per_key):
    """Weights over eight decades make every order of the sum visible."""
    print(f"case events of one key {per_key}", flush=True)
    n = 70
    m, o = _pair(oracle, ADEX, "RK4", n)
    rng = np.random.default_rng(per_key)
    for k in range(1, 6):
        tgt = np.repeat(np.array([0, 1, 63, 64, 69], np.int32), per_key)
        typ = rng.integers(0, 3, len(tgt)).astype(np.uint8)
        perm = rng.permutation(len(tgt))
        w = (10.0 ** rng.uniform(-6, 1.5, len(tgt))).astype(np.float32)
        _step(m, o, k, tgt[perm], typ[perm], w, pushes=1 + k % 3)
    _state(m, o)


def test_queue_grows(oracle):
    print("case queue grows", flush=True)
    n = 3000
    m, o = _pair(oracle, LIF, "Euler", n)
    rng = np.random.default_rng(5)
    for k, ne in enumerate((0, 1, 4095, 4097, 9000, 30_000, 10), 1):
        _step(m, o, k, rng.integers(0, n, ne).astype(np.int32), rng.integers(0, 2, ne).astype(np.uint8),
              rng.uniform(0, 0.3, ne).astype(np.float32), pushes=3)
    _state(m, o)


def test_many_spikes(oracle):
    """4,096 spikes go back with the compaction, more in a copy: updates on
    both sides of that and without spikes."""
    print("case many spikes", flush=True)
    n = 12_000
    m, o = _pair(oracle, LIF, "Euler", n)
    counts = []
    for k, hit in enumerate((0, 4095, 0, 4096, 4097, 12_000, 1), 1):
        v = o.state(0).astype(np.float32)
        v[:] = -65.0
        v[np.arange(hit) * (n // max(hit, 1))] = -40.0
        m.SetVectorNeuronState(0, v)
        o.set_state(0, v)
        z = np.zeros(0, np.int32)
        counts.append(_step(m, o, k, z, z.astype(np.uint8), z.astype(np.float32)))
    assert max(counts) > 4096 and 0 in counts
    _state(m, o)


@pytest.mark.parametrize("n", [1, 511, 512, 513, 1025])
@pytest.mark.parametrize("fp64", [False, True])
def test_bdf_tiles(oracle, n, fp64):
    print(f"case BDF tiles n={n} fp64={fp64}", flush=True)
    m, o = _pair(oracle, HH, "BDF", n, order=2, fp64=fp64)
    rng = np.random.default_rng(n)
    total = 0
    for k in range(1, 61):
        ne = n
        total += _step(m, o, k, rng.integers(0, n, ne).astype(np.int32), np.zeros(ne, np.uint8),
                       rng.uniform(0, 12, ne).astype(np.float32))
    assert total > 0
    _state(m, o)
