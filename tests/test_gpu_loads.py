"""Loads that are not finite, or whose squares leave the range of FP64, on the routes that the
direct factorisation takes: the result is that of the dense factorisations (which propagate
what is not a number and know no norms), and only the structure and load case concerned is
affected."""
from __future__ import annotations

import ctypes
import math
import warnings

import numpy as np
import pytest
import torch

from jaxsso_amd import _native as nat
from jaxsso_amd import workloads as wl
from jaxsso_amd.batch import StructureBatch
from jaxsso_amd.plan import FEPlan

pytestmark = pytest.mark.gpu

NOT_FINITE = [math.nan, math.inf, -math.inf]


def rel(a, b):
    return float(torch.linalg.norm(a - b) / torch.linalg.norm(b))


def shell(n, kx=1.0, ky=1.0, design=3):
    st = wl.shell_pinned_edges(n, 0.3 * n, 0.05 * n, design=design)
    st.prop_quads[:, 3], st.prop_quads[:, 4] = kx, ky
    return st


def plan_of(st, **kw):
    plan = FEPlan([0, st.n_node], st.cnct_beamcols, st.cnct_quads, st.known_id)
    return plan, plan.assemble(torch.tensor(st.crds), None, torch.tensor(st.prop_quads), **kw)


def free_dof(st):
    return int(np.setdiff1d(np.arange(st.ndof), st.known_id)[st.ndof // 3])


@pytest.mark.parametrize("value", NOT_FINITE)
@pytest.mark.parametrize("m", [1, 4, 5])
def test_dense_solve_of_a_load_that_is_not_finite(m, value):
    st = shell(9)
    plan, K = plan_of(st, export_K=True)
    F = np.random.default_rng(1).normal(size=(st.ndof, m))
    c = m // 2
    F[free_dof(st), c] = value
    f = torch.tensor(F[:, 0] if m == 1 else F, device="cuda")
    u, v = (plan.dense_solve(f, K=k).reshape(-1, m) for k in (None, K))   # v: the dense Cholesky
    assert torch.equal(torch.isfinite(u), torch.isfinite(v)) and not torch.isfinite(u[:, c]).any()
    for h in set(range(m)) - {c}:
        assert rel(u[:, h], v[:, h]) < 1e-9, h


# powers of two: the scaled problem has the scaled result, to the refinement's accuracy
@pytest.mark.parametrize("power", [-900, -565, -500, -450, 450, 530, 900])
@pytest.mark.parametrize("m", [1, 4])
def test_dense_solve_of_loads_whose_squares_leave_the_range(m, power):
    st = shell(9)
    plan, _ = plan_of(st)
    f = torch.tensor(np.random.default_rng(2).normal(size=(st.ndof, m)), device="cuda")
    u = plan.dense_solve(f)
    f[:, m - 1] *= 2.0 ** power                 # the other load cases stay ordinary
    v = plan.dense_solve(f)
    v[:, m - 1] *= 2.0 ** (-power // 2)
    v[:, m - 1] *= 2.0 ** (-power - -power // 2)
    for h in range(m):
        assert rel(v[:, h], u[:, h]) < 1e-9, h


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("value", NOT_FINITE)
def test_orthotropic_solve_of_a_load_that_is_not_finite(value, transpose):
    """One structure without a finite load in a batch: nothing finite comes out for it, the
    others are as without it, and it is not counted as converged (routes: refinement with the
    factor of the symmetric part; the iterative correction of a plan that chose its
    preconditioner)."""
    designs = [shell(6, 1.2, 0.8), shell(11, 1.2, 0.8), shell(8, 1.2, 0.8)]
    b = StructureBatch(designs)
    b.assemble()
    f = b.f[:, 0].contiguous()
    bad = f.clone()
    o = [6 * int(n) for n in b.node_off]
    bad[o[1] + free_dof(designs[1])] = value
    for route in ("direct", "iterative"):
        if route == "iterative":
            b.plan.nonsymmetric_route(2)
            b.plan.set_preconditioner("amg")
        good = b.plan.solve(f, transpose=transpose)
        assert b.plan.last_info["converged"] == 3
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", RuntimeWarning)
            u = b.plan.solve(bad, transpose=transpose)
        print(route, b.plan.last_info, flush=True)
        assert b.plan.last_info["converged"] == 2
        mid = torch.isfinite(u[o[1]:o[2]])
        assert not mid.any() if route == "direct" else not mid.all()
        for s in (0, 2):
            assert rel(u[o[s]:o[s + 1]], good[o[s]:o[s + 1]]) < 1e-9, (route, s)


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("power", [-900, -565, -500, 530, 900])
def test_orthotropic_solve_of_loads_whose_squares_leave_the_range(power, transpose):
    st = shell(9, 1.2, 0.8)
    plan, _ = plan_of(st)
    f = torch.tensor(st.nodal_loads, device="cuda")
    u = plan.solve(f, transpose=transpose)
    v = plan.solve(f * 2.0 ** power, transpose=transpose)
    v *= 2.0 ** (-power // 2)
    v *= 2.0 ** (-power - -power // 2)
    assert rel(v, u) < 1e-9


@pytest.mark.parametrize("preconditioner", [None, "amg", "block_jacobi"])
@pytest.mark.parametrize("value", NOT_FINITE)
def test_symmetric_batch_with_a_load_that_is_not_finite(preconditioner, value):
    designs = [wl.gridshell(6), shell(11), wl.gridshell(7)]
    b = StructureBatch(designs)
    b.assemble()
    f = b.f[:, 0].contiguous()
    bad = f.clone()
    o = [6 * int(n) for n in b.node_off]
    bad[o[1] + free_dof(designs[1])] = value
    good = b.plan.solve(f, preconditioner=preconditioner)
    with pytest.warns(RuntimeWarning):
        u = b.plan.solve(bad, preconditioner=preconditioner)
    info = b.plan.last_info
    assert info["converged"] == 2 and (info["levels"] > 0) == (preconditioner == "amg"), info
    mid = torch.isfinite(u[o[1]:o[2]])
    assert not mid.any() if preconditioner is None else not mid.all()
    for s in (0, 2):
        assert rel(u[o[s]:o[s + 1]], good[o[s]:o[s + 1]]) < 1e-8, s


def test_a_gradient_through_a_load_that_is_not_finite_is_not_finite():
    """The adjoint of an objective whose derivative is NaN, orthotropic and dense."""
    import jaxsso_amd.autograd as ag
    for st, opts in ((shell(7, 1.2, 0.8), ag.SolveOptions()), (shell(7), ag.SolveOptions(method="dense"))):
        plan = FEPlan([0, st.n_node], st.cnct_beamcols, st.cnct_quads, st.known_id)
        crds = torch.tensor(st.crds, device="cuda", requires_grad=True)
        pq, f = torch.tensor(st.prop_quads, device="cuda"), torch.tensor(st.nodal_loads, device="cuda")
        u = ag.displacement(plan, crds, None, pq, f, opts)
        w = torch.ones_like(u)
        w[free_dof(st)] = math.nan
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", RuntimeWarning)
            (g,) = torch.autograd.grad((u * w).sum(), crds)
        assert not torch.isfinite(g).all()


def test_a_plan_without_any_load_still_converges_to_zero():
    st = shell(9)
    plan, _ = plan_of(st)
    f = torch.zeros(st.ndof, dtype=torch.float64, device="cuda")
    info = nat.Info()
    u = torch.full_like(f, 7.0)
    nat.check(nat.lib().jsso_solve(plan._h, nat.ptr(f), nat.ptr(u), 1, nat.PREC["fp64"], 1e-10, 100,
                                   ctypes.byref(info), nat.stream_ptr()))
    assert info.converged == 1 and not u.any() and not plan.dense_solve(f).any()
