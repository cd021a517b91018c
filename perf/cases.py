"""The work this framework is asked to do, as measurable cases.

Kinds (each listed case is one of them, draw() spreads over the same ranges):

  plugin    the plug-in contract: one UpdateState with the step's input events
            pushed by the host and the spikes handed back
  network   a device-resident network advanced by a number of updates:
            Poisson-driven LIF, or a recurrent AdEx network in its settled state
  sweep     many independent AdEx networks as one grouped population
  circuit   the layered cerebellar circuit (granule BDF2, Golgi LIF, HH
            Purkinje cells with the FP64 Newton step, STDP)
  fit       one trace-fitting step: forward trace, squared error, gradients of
            every trained parameter
  session   a simulation built and advanced through Simulation_API

Outputs are the spikes of the pass (from the spike log, emptied after each
pass, in arrays of a fixed length; a sweep keeps the spike count only), the
populations' state rows and, where synapses are plastic, their weights.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import edlut_amd as E
from edlut_amd import _capi as C
from edlut_amd import simulation as S
from edlut_amd import workloads as W
from edlut_amd.adjoint import FitProblem, refractory_table
from edlut_amd.network import Network, binomial_thresholds, cerebellum_from_spec

DT = float(np.float32(1e-4))
LIF, ADEX, HH, GRANULE = ("LIFTimeDrivenModel_GPU", "AdExTimeDrivenModel_GPU", "HHTimeDrivenModel_GPU",
                          "EgidioGranuleCell_TimeDriven_GPU")
PLUGINS = {"lif": (LIF, "Euler"), "adex": (ADEX, "RK4"), "hh": (HH, "BDF"), "granule": (GRANULE, "BDF")}
SETTLE = 1000          # updates of a recurrent network before its first pass
BATCHES = 8            # event batches a plug-in program cycles through


def listed():
    return [
        # one step of the reference's CPU-sized network as a plug-in: 1,000 LIF
        # cells, the 125 input spikes 125,000 sources at 10 Hz send in 0.1 ms
        dict(name="plugin_lif_1000", kind="plugin", model="lif", n=1000, events=125, fp64=False),
        # a mid-sized conductance model, implicit method, FP64 Newton step
        dict(name="plugin_hh_bdf2_4099", kind="plugin", model="hh", n=4099, events=800, fp64=True),
        # the largest plug-in population: 1M AdEx, the spikes of a 5 Hz network
        # with in-degree 20 per neuron in a step
        dict(name="plugin_adex_1m", kind="plugin", model="adex", n=1_000_000, events=10_000, fp64=False),
        # the 1,000-cell LIF network with its 125,000 Poisson inputs, 25.6 ms
        dict(name="lif_poisson_1000", kind="network", model="lif", n=1000, fan_in=125, max_delay=50, steps=256),
        # a laptop-sized recurrent AdEx network, odd size
        dict(name="adex_20011", kind="network", model="adex", n=20_011, fan_in=100, max_delay=10, steps=128),
        # the headline network: 1M AdEx cells, in-degree 200, settled activity
        dict(name="adex_1m", kind="network", model="adex", n=1_000_000, fan_in=200, max_delay=10, steps=128),
        # parameter sweep: 512 networks of 1,000 to 20,000 cells
        dict(name="sweep_512", kind="sweep", networks=512, fan_in=100, max_delay=10, steps=32),
        # a small cerebellar circuit (odd granule count), where launches count
        dict(name="circuit_2501", kind="circuit", granule=2501, golgi=24, purkinje=5, mossy=500, steps=64),
        # the full-size cerebellar circuit
        dict(name="circuit_200k", kind="circuit", granule=200_000, golgi=2_000, purkinje=100, mossy=10_000, steps=16),
        # one fitting step of 256 LIF neurons over a second
        dict(name="fit_lif_256", kind="fit", model="lif", n=256, steps=10_000, n_syn=50),
        # one fitting step of 256 AdEx neurons over a second
        dict(name="fit_adex_256", kind="fit", model="adex", n=256, steps=10_000, n_syn=50),
        # 20 ms of a simulation written against Simulation_API
        dict(name="session_1000", kind="session", adex=800, lif=200, poisson=400, ms=20),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["plugin", "plugin", "network", "network", "sweep", "circuit", "fit", "fit", "session"])
    if kind == "plugin":
        model = rng.choice(["lif", "adex", "hh", "granule"])
        n = _log_int(rng, 100, {"lif": 1_000_000, "adex": 1_000_000, "hh": 50_000, "granule": 50_000}[model])
        return dict(kind=kind, model=model, n=n, events=max(1, int(n * rng.choice([0.002, 0.01, 0.1]))),
                    fp64=model == "hh" and rng.random() < 0.5)
    if kind == "network":
        if rng.random() < 0.4:
            return dict(kind=kind, model="lif", n=_log_int(rng, 100, 4000), fan_in=rng.randint(40, 125),
                        max_delay=rng.randint(10, 50), steps=rng.randint(64, 256))
        return dict(kind=kind, model="adex", n=_log_int(rng, 2000, 1_000_000), fan_in=rng.randint(50, 200),
                    max_delay=rng.randint(2, 16), steps=rng.randint(48, 128))
    if kind == "sweep":
        return dict(kind=kind, networks=_log_int(rng, 16, 512), fan_in=rng.randint(50, 100),
                    max_delay=rng.randint(4, 12), steps=rng.randint(16, 32))
    if kind == "circuit":
        g = _log_int(rng, 500, 200_000)
        return dict(kind=kind, granule=g, golgi=max(8, g // 100), purkinje=max(2, g // 2000),
                    mossy=max(50, g // 20), steps=rng.randint(16, 32) if g < 50_000 else 16)
    if kind == "fit":
        return dict(kind=kind, model=rng.choice(["lif", "adex"]), n=_log_int(rng, 16, 1024),
                    steps=_log_int(rng, 500, 10_000), n_syn=rng.randint(10, 80))
    return dict(kind=kind, adex=_log_int(rng, 100, 2000), lif=_log_int(rng, 50, 500), poisson=_log_int(rng, 100, 1000),
                ms=rng.choice([10, 20]))


# ---- inputs ---------------------------------------------------------------
class _Rows:
    """A population's state rows in device memory, without a copy."""

    def __init__(self, model):
        nv, nd, stride, p = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int64(0), ctypes.c_void_p()
        C.check(C.lib().edlut_population_layout(model.handle, C.byref(nv), C.byref(nd), C.byref(stride)))
        C.check(C.lib().edlut_population_device_state(model.handle, C.byref(p)))
        self.model = model
        self.__cuda_array_interface__ = dict(shape=(nv.value, model.size), typestr="<f4", version=2,
                                             data=(p.value, False), strides=(4 * stride.value, 4))


def _rows(model):
    return torch.as_tensor(_Rows(model), device="cuda")


def _lif_spec(case, seed):
    inh = case["fan_in"] // 5
    spec = W.lif_poisson(n=case["n"], n_exc=case["fan_in"] - inh, n_inh=inh, steps=case["steps"], seed=1 + seed)
    states, rate, (src, tgt, delay, typ, w) = spec.poisson[0]
    rng = np.random.default_rng(seed + 77)
    hi = case["max_delay"]
    delay = rng.integers(max(1, hi // 5), hi + 1, len(src)).astype(np.int32)
    spec.max_delay = hi
    spec.poisson[0] = (states, rate, (src, tgt, delay, typ, w))
    return spec


def _plugin_inputs(case, seed):
    """Initial membrane potentials and BATCHES event batches."""
    rng = np.random.default_rng(seed)
    n, ne = case["n"], case["events"]
    lo, hi = {"lif": (-65, -51), "adex": (-65, -51), "hh": (-70, -60), "granule": (-82, -70)}[case["model"]]
    v = rng.uniform(lo, hi, n).astype(np.float32)
    wmax = {"lif": 0.5, "adex": 8.0, "hh": 8.0, "granule": 1.5}[case["model"]]
    ev = []
    for _ in range(BATCHES):
        typ = (rng.random(ne) < 0.2).astype(np.uint8)
        ev.append((rng.integers(0, n, ne).astype(np.int32), typ, rng.uniform(0, wmax, ne).astype(np.float32)))
    return v, ev


def _fit_spec(case, seed):
    n_syn = case["n_syn"]
    return W.adjoint_fit(PLUGINS[case["model"]][0], n=case["n"], n_syn=n_syn, n_exc=n_syn - n_syn // 5,
                         steps=case["steps"], seed=5 + seed)


FIT_KEYS = ("g_leak", "e_leak", "tau_exc", "tau_inh", "weight")


def _fit_target(case, seed):
    """The recorded trace: a smooth membrane potential with noise."""
    rng = np.random.default_rng(seed + 991)
    return (-62.0 + 4.0 * rng.standard_normal((case["steps"], case["n"]), dtype=np.float32)).astype(np.float32)


def _session(case, seed):
    S.RandomGenerator.srand(seed % 30_000 + 1)
    sim = S.Simulation_API()
    rk4 = {"int_meth": {"name": "RK4", "step": 1e-4, "bdf_order": 1}}
    inp = sim.AddNeuronLayer(20, "InputSpikeNeuronModel")
    poi = np.array(sim.AddNeuronLayer(case["poisson"], "PoissonGeneratorDeviceVector", {"frequency": 40.0}))
    adex = np.array(sim.AddNeuronLayer(case["adex"], "AdExTimeDrivenModel_GPU", rk4, output_activity=True))
    lif = np.array(sim.AddNeuronLayer(case["lif"], "LIFTimeDrivenModel_GPU",
                                      {"int_meth": {"name": "Euler", "step": 1e-4}}, output_activity=True))
    rule = sim.AddLearningRule("STDP", {"max_LTP": 0.01, "tau_LTP": 0.02, "max_LTD": 0.012, "tau_LTD": 0.03})
    rng = np.random.default_rng(seed)

    def some(a, m):
        return a[rng.integers(0, len(a), m)]

    def delays(m):
        return (rng.integers(1, 11, m) * np.float32(1e-4)).astype(np.float32).tolist()

    m = 20 * case["adex"]
    sim.AddSynapticLayer(some(poi, m), some(adex, m), {"delay": delays(m), "weight": rng.uniform(2, 6, m).tolist()})
    m = 10 * case["adex"]
    sim.AddSynapticLayer(some(adex, m), some(adex, m), {"delay": delays(m), "type": 1, "weight": 1.0})
    m = 20 * case["lif"]
    sim.AddSynapticLayer(some(adex, m), some(lif, m),
                         {"delay": delays(m), "weight": 0.3, "wchange": rule, "max_weight": 1.0})
    m = 4 * len(inp)
    sim.AddSynapticLayer(some(np.array(inp), m), some(adex, m), {"delay": 0.001, "weight": 10.0})
    sim.Initialize()
    cells = rng.integers(0, len(inp), 100)
    slots = rng.choice(np.arange(10, 1000), 100, replace=False)
    order = np.argsort(slots)
    sim.AddExternalSpikeActivity(slots[order] * 1e-4 + 3e-5, cells[order] + inp[0])
    return sim


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "plugin":
        name, integ = PLUGINS[case["model"]]
        m = E.CreateNeuronModel(name, {"int_meth": E.integration_method(integ, DT, 2)})
        m.CheckSynapseType(0)
        m.CheckSynapseType(1)
        m.InitializeStates(case["n"])
        if case["fp64"]:
            m.SetNewtonFP64(True)
        v, ev = _plugin_inputs(case, seed)
        m.SetVectorNeuronState(0, v)
        st.update(model=m, events=ev, rows=_rows(m), k=0)
    elif kind == "network":
        if case["model"] == "lif":
            m, net = E.from_spec(_lif_spec(case, seed))
        else:
            m = E.CreateNeuronModel(ADEX, {"int_meth": E.integration_method("RK4", DT)})
            m.InitializeStates(case["n"])
            net = Network(m, case["max_delay"])
            net.generate_recurrent(case["fan_in"], 0.8, -1.0, 0.5, seed + 1)
            net.set_external(binomial_thresholds(100, 5.0 * DT), 0.65, seed * 1000003 + 11)
            net.run(SETTLE)
            net.clear_log()
        st.update(model=m, net=net, rows=_rows(m))
    elif kind == "sweep":
        spec = W.adex_sweep(n_networks=case["networks"], seed=4 + seed)
        m = E.CreateNeuronModel(ADEX, {"int_meth": E.integration_method("RK4", DT)})
        # the sizes are the sweep's, the parameters each seed's own
        m.InitializeGroups(W.adex_sweep(n_networks=case["networks"]).sizes, spec.params)
        net = Network(m, case["max_delay"])
        net.generate_recurrent(case["fan_in"], spec.exc_fraction, spec.w_mu, spec.w_sigma, spec.wiring_seed)
        net.set_external(*spec.ext)
        net.set_log_capacity(0)
        net.run(SETTLE)
        st.update(model=m, net=net, rows=_rows(m))
    elif kind == "circuit":
        g = case["granule"]
        spec = W.cerebellum(n_grc=g, n_goc=case["golgi"], n_pc=case["purkinje"], n_mf=case["mossy"],
                            k_goc=min(100, g // 10), k_pc=min(2000, g // 2), seed=3 + seed)
        models, nets, circuit = cerebellum_from_spec(spec)
        circuit.run(112)
        for n in nets:
            n.clear_log()
        st.update(models=models, nets=nets, circuit=circuit, rows=[_rows(m) for m in models])
    elif kind == "fit":
        spec = _fit_spec(case, seed)
        prob = FitProblem(spec.model, spec.params, spec.n, spec.steps, spec.syn_type, spec.events)
        x = [torch.tensor(spec.start[k], device="cuda", requires_grad=True) for k in FIT_KEYS]
        st.update(prob=prob, x=x, target=torch.from_numpy(_fit_target(case, seed)).cuda())
    else:
        sim = _session(case, seed)
        sim.RunSimulation(0.01)
        sim.GetSpikeActivity()
        st.update(sim=sim, t=0.01, rows=[_rows(m) for m in sim.models.values()])
    return st


# ---- one pass ---------------------------------------------------------------
def _spikes(net, cap):
    """The logged spikes, ascending by update, in arrays of `cap` entries."""
    out = np.full((2, cap), -1, np.int32)
    step, idx = net.spikes()
    net.clear_log()
    m = min(len(step), cap)
    out[0, :m], out[1, :m] = step[:m], idx[:m]
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "plugin":
        m = state["model"]
        state["k"] += 1
        m.ProcessInputSpikes(*state["events"][state["k"] % BATCHES])
        m.UpdateState(step=state["k"])
        idx = m.GetInternalSpikeIndexs()[: case["n"] // 64 + 64]
        spikes = np.full(case["n"] // 64 + 64, -1, np.int32)
        spikes[: len(idx)] = idx
        return {"spikes": spikes, "state": state["rows"]}
    if kind == "network":
        net = state["net"]
        net.run(case["steps"])
        return {"spikes": _spikes(net, case["n"] // 8 + 8192), "state": state["rows"]}
    if kind == "sweep":
        net = state["net"]
        net.run(case["steps"])
        return {"count": net.spike_count(), "state": state["rows"]}
    if kind == "circuit":
        state["circuit"].run(case["steps"])
        return {"state": state["rows"], "weight": state["nets"][2].synapses(0)[2],
                "spikes": [_spikes(net, m.size // 2 + 1024) for net, m in zip(state["nets"], state["models"])]}
    if kind == "fit":
        x = state["x"]
        v = state["prob"].simulate(*x)
        loss = ((v - state["target"]) ** 2).mean()
        return {"v": v, "grads": torch.autograd.grad(loss, x)}
    sim = state["sim"]
    state["t"] += case["ms"] * 1e-3
    sim.RunSimulation(state["t"])
    t, cells = sim.GetSpikeActivity()
    cap = 8 * (case["adex"] + case["lif"])
    out = np.full((2, cap), -1.0)
    m = min(len(t), cap)
    out[0, :m], out[1, :m] = t[:m], cells[:m]
    return {"spikes": out, "state": state["rows"]}


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    kind, steps = case["kind"], case.get("steps", 1)
    if kind == "plugin":
        # rows read and written (BDF: two history levels too), events once
        rows, fl = {"lif": (3, 20), "adex": (4, 140), "hh": (6, 3000), "granule": (17, 30_000)}[case["model"]]
        hist = {"hh": 4 * 3 * (8 if case["fp64"] else 4), "granule": 15 * 3 * 4}.get(case["model"], 0)
        return {"bytes": case["n"] * (8 * rows + 2 * hist) + 9 * case["events"], "flops": case["n"] * fl}
    if kind == "network":
        if case["model"] == "lif":
            gens = case["n"] * case["fan_in"]
            return {"bytes": steps * (case["n"] * 32 + gens * 8), "flops": steps * (case["n"] * 20 + gens * 6)}
        return {"bytes": steps * case["n"] * 32, "flops": steps * case["n"] * 160}
    if kind == "sweep":
        n = case["networks"] * 5650           # mean size of the clipped lognormal
        return {"bytes": steps * n * 32, "flops": steps * n * 160}
    if kind == "circuit":
        g = case["granule"]
        return {"bytes": steps * g * (17 * 8 + 15 * 3 * 8), "flops": steps * g * 30_000}
    if kind == "fit":
        per, fl = (8, 70) if case["model"] == "lif" else (8, 500)
        return {"bytes": case["n"] * (steps * per + case["n_syn"] * 8), "flops": case["n"] * steps * fl}
    n = case["adex"] + case["lif"]
    return {"bytes": case["ms"] * 10 * (n * 32 + case["poisson"] * 8), "flops": case["ms"] * 10 * n * 160}


def tolerance(case):
    # the simulation's contract is the reference's float arithmetic in its
    # order of events: every implementation of it gives the same bits
    if case["kind"] != "fit":
        return "exact"
    # forward and adjoint in 32 bits along the same spikes: LIF gradients lie
    # 1e-6 to 2e-6 from 64 bits; the AdEx upswings before a spike amplify the
    # rounding of the adjoint sweep (up to 1e-4 along one trajectory)
    return {"rel": 1e-5} if case["model"] == "lif" else {"rel": 4e-4}


# ---- the same in 64 bits -----------------------------------------------------
def _params(name):
    return {k: float(np.float32(v)) for k, v in E.REGISTRY[name].PARAMS}


DT_MS = float(np.float32(np.float32(1e-4) * np.float32(1000.0)))


def _exact_plugin(case, seed):
    if case["model"] == "granule":
        return None
    name, _ = PLUGINS[case["model"]]
    p = _params(name)
    v0, ev = _plugin_inputs(case, seed)
    n = case["n"]
    v = v0.astype(np.float64)
    tgt, typ, w = ev[1]
    ge = np.bincount(tgt[typ == 0], w[typ == 0].astype(np.float64), n)
    gi = np.bincount(tgt[typ == 1], w[typ == 1].astype(np.float64), n)
    h = DT_MS

    def cur(v, ge, gi):
        return ge * (p["e_exc"] - v) + gi * (p["e_inh"] - v)

    def decayed(ge, gi, t):
        return ge * math.exp(-t / p["tau_exc"]), gi * math.exp(-t / p["tau_inh"])

    z = np.zeros(n)
    if case["model"] == "lif":
        v = v + h * (cur(v, ge, gi) + p["g_leak"] * (p["e_leak"] - v)) / p["c_m"]
        v = np.where(v > p["v_thr"], p["e_leak"], v)
        ge, gi = decayed(ge, gi, h)
        rows = [v, ge, gi, z, z]
    elif case["model"] == "adex":
        def f(v, u, ge, gi):
            return ((p["g_leak"] * (p["e_leak"] - v) + p["g_leak"] * p["thr_slo_fac"] *
                     np.exp((v - p["v_thr"]) / p["thr_slo_fac"]) - u + cur(v, ge, gi)) / p["c_m"],
                    (p["a"] * (v - p["e_leak"]) - u) / p["tau_w"])
        u = np.zeros(n)
        k1 = f(v, u, ge, gi)
        gm = decayed(ge, gi, h / 2)
        k2 = f(v + k1[0] * h / 2, u + k1[1] * h / 2, *gm)
        k3 = f(v + k2[0] * h / 2, u + k2[1] * h / 2, *gm)
        g2 = decayed(ge, gi, h)
        k4 = f(v + k3[0] * h, u + k3[1] * h, *g2)
        v = v + (k1[0] + 2 * (k2[0] + k3[0]) + k4[0]) * h / 6
        u = u + (k1[1] + 2 * (k2[1] + k3[1]) + k4[1]) * h / 6
        rows = [v, u, g2[0], g2[1], z, z]
    else:
        # the first BDF step is an implicit Euler step: Newton to convergence
        def rates(v):
            x = v - p["v_thr"]
            am = 0.32 * (13 - x) / np.expm1((13 - x) / 4)
            bm = 0.28 * (x - 40) / np.expm1((x - 40) / 5)
            ah, bh = 0.128 * np.exp((17 - x) / 18), 4 / (1 + np.exp((40 - x) / 5))
            an, bn = 0.032 * (15 - x) / np.expm1((15 - x) / 5), 0.5 * np.exp((10 - x) / 40)
            return am, bm, ah, bh, an, bn

        am, bm, ah, bh, an, bn = rates(np.array([p["e_leak"]]))
        m0, h0, n0 = am / (am + bm), ah / (ah + bh), an / (an + bn)
        ge, gi = decayed(ge, gi, h)

        def gates(v):
            am, bm, ah, bh, an, bn = rates(v)
            return ((m0 + h * am) / (1 + h * (am + bm)), (h0 + h * ah) / (1 + h * (ah + bh)),
                    (n0 + h * an) / (1 + h * (an + bn)))

        def res(x):
            m, hh, nn = gates(x)
            return x - v - h * (cur(x, ge, gi) + p["g_leak"] * (p["e_leak"] - x) +
                                p["g_na"] * m ** 3 * hh * (p["e_na"] - x) +
                                p["g_kd"] * nn ** 4 * (p["e_k"] - x)) / p["c_m"]

        x = v.copy()
        for _ in range(40):
            e = 1e-6
            x = x - res(x) / ((res(x + e) - res(x - e)) / (2 * e))
        rows = [x, *gates(x), ge, gi, z, z]
    return {"spikes": None, "state": np.stack(rows)}


def _exact_lif(case, seed):
    """The Poisson-driven LIF network: the generators' integer sequences, the
    membrane and conductances in 64 bits."""
    spec = _lif_spec(case, seed)
    states, rate, (src, tgt, delay, typ, w) = spec.poisson[0]
    p = _params(LIF)
    n, D = case["n"], case["max_delay"]
    refr = refractory_table(1e-4, p["tau_ref"]).astype(np.float64)
    x = states.astype(np.uint64)
    v = np.full(n, p["e_leak"])
    g = np.zeros((2, n))
    since = np.full(n, 1 << 20)
    ring = np.zeros((D + 2, 2, n))
    dec = np.array([[math.exp(-DT_MS / p["tau_exc"])], [math.exp(-DT_MS / p["tau_inh"])]])
    frate, step_s = float(np.float32(rate)), float(np.float32(np.float32(0.1) / np.float32(1000.0)))
    for k in range(1, case["steps"] + 1):
        x = (x * np.uint64(1103515245) + np.uint64(12345)) & np.uint64(0x7FFFFFFF)
        u = x.astype(np.float32) / np.float32(2147483647.0)
        hit = np.nonzero(frate * step_s > u.astype(np.float64))[0]
        slot = k % (D + 2)
        g += ring[slot]
        ring[slot] = 0.0
        np.add.at(ring, ((k + delay[hit] + 1) % (D + 2), typ[hit].astype(np.int64), tgt[hit]), w[hit].astype(np.float64))
        frac = np.where(since < len(refr), np.maximum(refr[np.minimum(since, len(refr) - 1)], 0.0), 1.0)
        dv = (g[0] * (p["e_exc"] - v) + g[1] * (p["e_inh"] - v) + p["g_leak"] * (p["e_leak"] - v)) / p["c_m"]
        v = v + DT_MS * frac * dv
        g = np.where(g < 1e-9, 0.0, g * dec)
        fired = v > p["v_thr"]
        v[fired] = p["e_leak"]
        since = np.where(fired, 0, since + 1)
    z = np.zeros(n)
    return {"spikes": None, "state": np.stack([v, g[0], g[1], z, z])}


def _exact_fit(case, seed):
    """LIF trace and gradients in 64 bits by torch's autograd, a segment of
    updates at a time (the spikes' positions carry no gradient)."""
    if case["model"] != "lif" or case["steps"] * (1 + case["n"] / 2000) > 12_000:
        return None
    spec = _fit_spec(case, seed)
    p = _params(LIF)
    refr = torch.from_numpy(np.maximum(refractory_table(1e-4, p["tau_ref"]).astype(np.float64), 0.0))
    n, steps = spec.n, spec.steps
    gl, el, te, ti, w = [torch.tensor(spec.start[k], dtype=torch.float64, requires_grad=True) for k in FIT_KEYS]
    ptr, ev_step, ev_syn = (torch.from_numpy(a.astype(np.int64)) for a in spec.events)
    owner = torch.repeat_interleave(torch.arange(n), ptr[1:] - ptr[:-1])
    order = torch.argsort(ev_step, stable=True)
    owner, ev_syn, ev_step = owner[order], ev_syn[order], ev_step[order]
    at = torch.searchsorted(ev_step, torch.arange(steps + 2)).tolist()
    inh = torch.from_numpy(spec.syn_type.astype(np.int64))[owner, ev_syn]
    target = torch.from_numpy(_fit_target(case, seed)).double()
    h = DT_MS

    def advance(x, gl, el, te, ti, w, k0, k1):
        v, ge, gi, since = x
        ce, ci = torch.exp(-h / te), torch.exp(-h / ti)
        out = []
        for k in range(k0, k1):
            a, b = at[k], at[k + 1]
            if b > a:
                wk, o, t = w[owner[a:b], ev_syn[a:b]], owner[a:b], inh[a:b].double()
                ge = ge.index_add(0, o, wk * (1 - t))
                gi = gi.index_add(0, o, wk * t)
            frac = torch.where(since < len(refr), refr[since.clamp(max=len(refr) - 1)], torch.ones(n).double())
            v = v + h * frac * ((ge * (p["e_exc"] - v) + gi * (p["e_inh"] - v) + gl * (el - v)) / p["c_m"])
            ge = torch.where(ge < 1e-9, torch.zeros_like(ge), ge * ce)
            gi = torch.where(gi < 1e-9, torch.zeros_like(gi), gi * ci)
            fired = v > p["v_thr"]
            v = torch.where(fired, el, v)
            since = torch.where(fired, 0, (since + 1).clamp(max=1 << 20))
            out.append(v)
        return (v, ge, gi, since), torch.stack(out)

    z = torch.zeros(n, dtype=torch.float64)
    x, trace = (el, z, z, torch.full((n,), 1 << 20)), []
    total = None
    for k0 in range(1, steps + 1, 500):
        x, v = advance(x, gl, el, te, ti, w, k0, min(k0 + 500, steps + 1))
        trace.append(v)
    v = torch.cat(trace)
    total = ((v - target) ** 2).mean()
    return {"v": v.detach().numpy(), "grads": [t.numpy() for t in torch.autograd.grad(total, (gl, el, te, ti, w))]}


def exact(case, seed):
    """Recurrent networks, sweeps, circuits and sessions have no 64-bit
    counterpart: a rounding moves a spike, and the run with it."""
    if case["kind"] == "plugin":
        return _exact_plugin(case, seed)
    if case["kind"] == "network" and case["model"] == "lif":
        return _exact_lif(case, seed)
    if case["kind"] == "fit":
        return _exact_fit(case, seed)
    return None
