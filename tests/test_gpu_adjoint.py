"""The adjoint kernels over several load cases and element counts around a workgroup (64
quads, 256 beam cases), and the backward pass of evaluations that share a plan."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from jaxsso_amd import autograd
from jaxsso_amd import workloads as wl
from jaxsso_amd.plan import FEPlan
from test_gpu_direct import ribbed

pytestmark = pytest.mark.gpu


def plan_of(st):
    return FEPlan([0, st.n_node], st.cnct_beamcols, st.cnct_quads, st.known_id)


def inputs(st):
    return [torch.tensor(a, device="cuda") for a in (st.crds, st.prop_beamcols, st.prop_quads)]


@pytest.mark.parametrize("n", [2, 4, 8, 9])   # 4, 16, 64 and 81 quads
@pytest.mark.parametrize("general", [False, True])
def test_load_cases_of_one_call_match_calls_of_one(n, general):
    """The same arithmetic per (element, load case): the same bits; lambda = u/2 passed as a
    tensor differs from the form that does not read it by rounding only."""
    st = wl.shell_pinned_edges(n, 2.0, 0.4, design=1)
    st.crds[:, 2] += np.random.default_rng(n).normal(0.0, 0.02, st.n_node)
    plan, (crds, pb, pq) = plan_of(st), inputs(st)
    plan.assemble(crds, pb, pq)
    g = torch.Generator(device="cuda").manual_seed(n)
    u = torch.randn(st.ndof, 3, dtype=torch.float64, device="cuda", generator=g)
    lam = torch.randn(u.shape, dtype=torch.float64, device="cuda", generator=g) if general else None
    dc, _, dq = plan.adjoint(crds, pb, pq, u, lam=lam, lam_scale=0.5)
    for h in range(3):
        one = u[:, h].contiguous()
        ec, _, eq = plan.adjoint(crds, pb, pq, one, lam=lam[:, h].contiguous() if general else None, lam_scale=0.5)
        assert torch.equal(dc[..., h], ec) and torch.equal(dq[..., h], eq)
        if not general:
            fc, _, fq = plan.adjoint(crds, pb, pq, one, lam=0.5 * one)
            # both are exact derivatives of up to 4 quads' energies a node: some 1e3 roundings
            assert (fc - ec).abs().max() < 1e-12 * ec.abs().max() and (fq - eq).abs().max() < 1e-12 * eq.abs().max()


def test_backward_after_the_plan_was_assembled_again():
    """Gradients of two evaluations on one plan, taken in either order and twice, are those
    of the evaluations on plans of their own (compliance and a displacement objective)."""
    st = ribbed(9)
    shared = plan_of(st)
    f = torch.tensor(st.nodal_loads, device="cuda")
    wgt = torch.linspace(0.5, 1.5, st.ndof, dtype=torch.float64, device="cuda")

    def evaluate(plan, scale, which):
        crds, pb, pq = inputs(st)
        crds[:, 2] *= scale
        crds.requires_grad_(True)
        val = autograd.compliance(plan, crds, pb, pq, f)[0] if which else \
            (wgt * autograd.displacement(plan, crds, pb, pq, f)).sum()
        return val, crds

    def grad(v):
        return torch.autograd.grad(v[0], v[1], retain_graph=True)[0]

    for which in (True, False):
        own = [grad(evaluate(plan_of(st), s, which)) for s in (1.0, 1.4)]
        a, b = evaluate(shared, 1.0, which), evaluate(shared, 1.4, which)
        for v, ref in ((a, own[0]), (b, own[1]), (b, own[1]), (a, own[0])):
            # both solve to 1e-10 of the load
            assert (grad(v) - ref).abs().max() < 1e-7 * ref.abs().max(), which
