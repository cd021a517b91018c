"""Trace fitting at the edges of the backward pass's segments: populations and
runs that end inside a wave or a segment, checkpoint spacings below the
longest segment, steps with more than two events of one type, and runs whose
segments take several launches.
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
    """16,384 neurons over 1,600 steps need two backward launches.  They are
    256 copies of 64 neurons: each copy's gradients equal the 64-neuron
    problem's (one launch) but for the grouping of double sums rounded to
    float, and those of its weights, summed in float in the same order, bit
    for bit up to the adjoint state that enters the second launch (double)."""
    n, copies, steps = 64, 256, 1600
    print(f"case several launches {model}", flush=True)
    spec, prob, x = _problem(model, n, steps, 100, 20.0)
    ptr, st, sy = spec.events
    big = np.concatenate([[0]] + [ptr[1:] + c * ptr[-1] for c in range(copies)]).astype(np.int32)
    many = FitProblem(model, spec.params, n * copies, steps, np.tile(spec.syn_type, (copies, 1)),
                      (big, np.tile(st, copies), np.tile(sy, copies)))
    y = [t.repeat(copies) if t.dim() == 1 else t.repeat(copies, 1) for t in x]
    gv = torch.randn(steps, n, device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    v = prob.forward_raw(*x)
    gp, gw = prob.backward_raw(*x, gv)
    vm = many.forward_raw(*y)
    gpm, gwm = many.backward_raw(*y, gv.repeat(1, copies))
    assert torch.equal(vm.view(steps, copies, n)[:, 0], v) and torch.equal(vm.view(steps, copies, n)[:, -1], v)
    for a, b in ((gpm.view(4, copies, n), gp[:, None]), (gwm.view(copies, n, -1), gw[None])):
        assert float((a - b).abs().max()) <= 1e-6 * float(b.abs().max())
