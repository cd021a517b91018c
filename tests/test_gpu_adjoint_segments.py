"""Trace fitting at the edges of the backward pass's segments: populations and
runs that end inside a wave or a segment, checkpoint spacings below the
longest segment, steps with more than two events of one type, runs whose
segments take several launches, and checkpoints further apart than segments.
"""
import numpy as np
import pytest
import torch

from edlut_amd import workloads
from edlut_amd.adjoint import FitProblem, refractory_table

pytestmark = pytest.mark.gpu
LIF, ADEX = "LIFTimeDrivenModel_GPU", "AdExTimeDrivenModel_GPU"
KEYS = ("g_leak", "e_leak", "tau_exc", "tau_inh", "weight")


def _problem(model, n, steps, ckpt, rate, seed=3):
    spec = workloads.adjoint_fit(model, n=n, steps=steps, n_syn=20, n_exc=15, rate=rate, seed=seed)
    prob = FitProblem(model, spec.params, n, steps, spec.syn_type, spec.events, checkpoint=ckpt)
    x = [torch.tensor(spec.start[k], dtype=torch.float32, device="cuda") for k in KEYS]
    return spec, prob, x


@pytest.mark.parametrize("model", [LIF, ADEX])
@pytest.mark.parametrize("n,steps,ckpt,rate", [(1, 1, 100, 3000.0), (3, 31, 100, 200.0), (64, 32, 100, 20.0),
                                               (65, 33, 100, 20.0), (7, 200, 1, 20.0), (130, 321, 7, 50.0),
                                               (33, 500, 100, 1500.0)])
def test_segment_edges(oracle, model, n, steps, ckpt, rate):
    """Gradients against the FP64 adjoint along the same trajectory, to the
    float adjoint's 1e-4 (a rate of 1,500 Hz puts three or more events of one
    type into most steps)."""
    print(f"case segments {model} n={n} steps={steps} ckpt={ckpt} rate={rate}", flush=True)
    spec, prob, x = _problem(model, n, steps, ckpt, rate)
    refr = refractory_table(1e-4, float(spec.params[7])) if model == LIF else None
    o = oracle.FitOracle(model, spec.params, n, steps, spec.syn_type, spec.events, refr)
    v, spk, traj, since = prob.forward_raw(*x, spikes=True, trajectory=True)
    gv = torch.randn(steps, n, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    gp, gw = prob.backward_raw(*x, gv)
    torch.cuda.synchronize()
    vf, _ = o.forward(*[spec.start[k] for k in KEYS], fp64=False)
    if steps <= 33:    # before any spike the two forwards differ by their libms' expf only
        assert np.allclose(v.cpu().numpy(), vf, rtol=1e-5, atol=1e-5)
    rp, rw = o.backward_along(*[spec.start[k] for k in KEYS], gv.cpu().numpy().astype(np.float64),
                              traj.cpu().numpy(), spk.cpu().numpy(), since.cpu().numpy())
    for a, b in zip([*gp.cpu().numpy(), gw.cpu().numpy()], [*rp, rw]):
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b) + 1e-12


@pytest.mark.parametrize("model", [LIF, ADEX])
def test_several_launches(model):
    """16,384 neurons over 1,600 steps need two backward launches."""
    print(f"case several launches {model}", flush=True)
    _copies(model, 256, 1600, 100)


def _copies(model, copies, steps, ckpt):
    """Copies of 64 neurons in one problem against the 64-neuron problem (one
    launch, a checkpoint for every segment).  The same V trace bit for bit; the
    gradients are the same terms, grouped into launches otherwise and summed in
    double (parameters) or from an adjoint state that is the same to double's
    rounding (weights) before they are rounded to float: a unit in the last
    place or two of the largest."""
    n = 64
    spec, prob, x = _problem(model, n, steps, 100, 20.0)
    ptr, st, sy = spec.events
    big = np.concatenate([[0]] + [ptr[1:] + c * ptr[-1] for c in range(copies)]).astype(np.int32)
    many = FitProblem(model, spec.params, n * copies, steps, np.tile(spec.syn_type, (copies, 1)),
                      (big, np.tile(st, copies), np.tile(sy, copies)), checkpoint=ckpt)
    y = [t.repeat(copies) if t.dim() == 1 else t.repeat(copies, 1) for t in x]
    gv = torch.randn(steps, n, device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    v = prob.forward_raw(*x)
    gp, gw = prob.backward_raw(*x, gv)
    vm = many.forward_raw(*y)
    gpm, gwm = many.backward_raw(*y, gv.repeat(1, copies))
    assert torch.equal(vm.view(steps, copies, n)[:, 0], v) and torch.equal(vm.view(steps, copies, n)[:, -1], v)
    for a, b in ((gpm.view(4, copies, n), gp[:, None]), (gwm.view(copies, n, -1), gw[None])):
        assert float((a - b).abs().max()) <= 1e-6 * float(b.abs().max())


@pytest.mark.parametrize("model", [LIF, ADEX])
@pytest.mark.parametrize("steps,ckpt", [(1600, 100), (1650, 170), (1600, 5000)])
def test_checkpoints_apart(model, steps, ckpt):
    """230,400 neurons: a state every 32 steps would take more than 256 MB, so
    one is kept for every 3 segments, for 5 (with segments and steps left over)
    and for the whole run (its states then take several launches' segments)."""
    print(f"case checkpoints apart {model} steps={steps} ckpt={ckpt}", flush=True)
    _copies(model, 3600, steps, ckpt)


def test_checkpoint_memory():
    """50,000 neurons over 20,000 steps: a state every 32 steps takes 750 MB, one
    every 960 steps 25 MB."""
    print("case checkpoint memory", flush=True)
    n, steps = 50_000, 20_000
    spec = workloads.adjoint_fit(LIF, n=1, steps=1, n_syn=1, n_exc=1, rate=1.0, seed=1)
    used = []
    for ckpt in (32, 1000):
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        prob = FitProblem(LIF, spec.params, n, steps, np.zeros((n, 1), np.uint8),
                          (np.zeros(n + 1, np.int32), np.zeros(1, np.int32), np.zeros(1, np.int32)), checkpoint=ckpt)
        used.append(free - torch.cuda.mem_get_info()[0])
        prob.close()
    assert used[0] - used[1] > 600 << 20, used
