"""Which calls the direct solve serves, and what of it a plan keeps."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from jaxsso_amd import _native as nat
from jaxsso_amd import workloads as wl
from jaxsso_amd.batch import StructureBatch
from jaxsso_amd.plan import FEPlan

pytestmark = pytest.mark.gpu


def shell(n, kx=1.0, ky=1.0):
    st = wl.shell_pinned_edges(n, 0.3 * n, 0.05 * n, design=3)
    st.prop_quads[:, 3], st.prop_quads[:, 4] = kx, ky
    return st


def plan_of(st):
    plan = FEPlan([0, st.n_node], st.cnct_beamcols, st.cnct_quads, st.known_id)
    plan.assemble(torch.tensor(st.crds), None, torch.tensor(st.prop_quads))
    return plan


def test_a_plan_tells_how_it_solves():
    one, two = StructureBatch([shell(24)]), StructureBatch([shell(24), shell(24)])
    assert one.plan.direct_info()["taken"] is None and one.plan.direct_info()["begun"] == 0
    for _ in range(2):
        one.solve(), one.solve(assemble=False), two.solve()
    a, b = one.plan.direct_info(), two.plan.direct_info()
    print(a, b, flush=True)
    assert a["taken"] and a["factorisations"] == 2 and a["begun"] == a["finished"] == 4
    assert 0 < a["max_front"] == b["max_front"] <= 2300 and a["max_front"] % 6 == 0
    # the two structures of one pattern: twice the operations and the memory
    assert b["operations"] == 2 * a["operations"] and b["bytes"] == 2 * a["bytes"] > 0
    large = FEPlan([0, 301 ** 2], np.zeros((0, 2), np.int32), shell(300).cnct_quads, [0, 1, 2])
    assert large.direct_info()["taken"] is None


@pytest.mark.parametrize("transpose", [False, True])
def test_the_iterative_correction_runs_its_inner_solver_alone(transpose):
    """K so far from its symmetric part (spectral radius of I - S^-1 K about 0.65) that the
    refinement with the factor of S, which wants 0.5, hands over to the iterative correction:
    the direct solve is not begun again for its inner solves."""
    plan = plan_of(shell(12, 14.0, 1.0))
    plan.nonsymmetric_route(2)
    f = torch.tensor(shell(12).nodal_loads, device="cuda")
    u = plan.solve(f, transpose=transpose)
    info, direct = plan.last_info, plan.direct_info()
    print(info, direct, flush=True)
    assert info["converged"] == 1 and info["replacements"] > 3 and info["iterations"] > info["replacements"]
    assert direct["factorisations"] == direct["begun"] == 1 and direct["finished"] == 0
    plan.nonsymmetric_route(1)
    dense = plan.solve(f, transpose=transpose)
    assert float(torch.linalg.norm(u - dense) / torch.linalg.norm(dense)) < 1e-8


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("ratio,route", [(1.5, 0), (1.5, 2), (14.0, 2)])
def test_a_result_over_the_right_hand_side_of_a_non_symmetric_solve(ratio, route, transpose):
    """u = f in memory, u half over f, and apart: the same u on each route (refinement with the
    factor of the symmetric part, iterative correction; two load cases)."""
    st = shell(9, ratio, 1.0)
    plan = plan_of(st)
    n = 2 * st.ndof
    rng = np.random.default_rng(4)
    f = torch.tensor(st.nodal_loads[:, None] * rng.uniform(0.5, 2.0, (st.ndof, 2)), device="cuda").reshape(-1)
    plan.nonsymmetric_route(1)
    ref = plan.solve(f.reshape(-1, 2), transpose=transpose).reshape(-1)
    plan.nonsymmetric_route(route)
    entry = nat.lib().jsso_solve_transpose if transpose else nat.lib().jsso_solve
    for gap in (0, n // 2, -(n // 2), n):
        info = nat.Info()
        both = torch.zeros(3 * n, dtype=torch.float64, device="cuda")
        fv, uv = both[n:2 * n], both[n + gap:2 * n + gap]
        fv.copy_(f)
        nat.check(entry(plan._h, nat.ptr(fv), nat.ptr(uv), 2, nat.PREC["fp64"], 1e-11, 10000, ctypes.byref(info),
                        nat.stream_ptr()))
        print(ratio, route, gap, info.as_dict(), flush=True)
        assert info.converged == 2 and info.replacements > 0
        assert float(torch.linalg.norm(uv - ref) / torch.linalg.norm(ref)) < 1e-8, gap


def test_ensure_assembled_without_an_assembly_id():
    """The call with inputs alone makes the plan hold their assembly."""
    a, b = shell(9), shell(9, 1.5, 1.0)
    plan = plan_of(a)
    f = torch.tensor(a.nodal_loads, device="cuda")
    u = plan.solve(f)
    first = plan.assembly_id
    inputs = torch.tensor(a.crds, device="cuda"), None, torch.tensor(a.prop_quads, device="cuda")
    plan.assemble(torch.tensor(b.crds), None, torch.tensor(b.prop_quads))
    assert not torch.equal(plan.solve(f), u)
    now = plan.ensure_assembled(*inputs)
    assert now == plan.assembly_id > first and torch.equal(plan.solve(f), u)
    assert plan.ensure_assembled(*inputs, now) == now


def test_a_plan_holds_the_memory_of_the_inputs_that_it_assembles():
    """Inputs made on the current stream, assembled on another one and dropped: their memory
    is not handed out while the assembly may still read it."""
    st = shell(20)
    plan = plan_of(st)
    f = torch.tensor(st.nodal_loads, device="cuda")
    u = plan.solve(f)
    side = torch.cuda.Stream()
    crds, pq = torch.tensor(st.crds, device="cuda"), torch.tensor(st.prop_quads, device="cuda")
    held = {crds.data_ptr(), pq.data_ptr()}
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        plan.assemble(crds, None, pq)
    shapes = crds.shape, pq.shape
    del crds, pq
    new = [torch.zeros(sh, dtype=torch.float64, device="cuda") for sh in shapes for _ in range(4)]
    assert not held & {t.data_ptr() for t in new}
    side.synchronize()
    assert torch.equal(plan.solve(f), u)


def test_a_choice_of_the_iterative_solve_can_be_taken_back():
    """preconditioner="amg" for one call, a kept AMG hierarchy given up, and a chosen
    preconditioner taken back: the plan solves directly again; a choice that is not taken back
    stays."""
    st = shell(12)
    plan = plan_of(st)
    f = torch.tensor(st.nodal_loads, device="cuda")

    def direct(**kw):
        plan.solve(f, **kw)
        return plan.last_info["levels"] == 0 and plan.last_info["iterations"] <= 6

    assert direct() and not direct(preconditioner="amg") and direct()
    assert plan.preconditioner == "amg"
    plan.amg_reuse(2)
    assert not direct() and not direct(preconditioner="amg") and not direct()
    plan.amg_reuse(0)
    assert direct()
    for name in ("amg", "block_jacobi"):
        plan.set_preconditioner(name)
        assert not direct() and not direct(preconditioner=name) and not direct() and plan.preconditioner == name
        plan.set_preconditioner(None)
        assert direct()
    assert not direct(preconditioner="block_jacobi") and not direct() and plan.preconditioner == "block_jacobi"
    with pytest.raises(ValueError):
        plan.set_preconditioner("ilu")
    with pytest.raises(RuntimeError):
        nat.check(nat.lib().jsso_plan_set_preconditioner(plan._h, 7))


@pytest.mark.parametrize("nrhs", [1, 2, 3, 4])
def test_plans_of_one_pattern_give_the_same_bits(nrhs):
    """The order of the residual's sums is the pattern's, not a timing's: plans made one after
    the other choose the same waves per slice and return the same bits after two steps."""
    st = shell(6)
    f = torch.tensor(np.random.default_rng(3).normal(size=(st.ndof, nrhs)), device="cuda")
    first = None
    for _ in range(24):
        plan = plan_of(st)
        u = plan.solve(f, tol=1e-16)
        waves = plan.cg_tuning("fp64", nrhs)
        assert plan.last_info["iterations"] >= 2 and plan.last_info["waves_per_slice"] == waves
        first = first or (waves, u)
        assert waves == first[0] and torch.equal(u, first[1])


def test_a_mesh_past_the_limit_of_the_fronts_takes_the_iterative_route():
    st = wl.shell_pinned_edges(270, 27.0, 3.0, design=3)
    plan = plan_of(st)
    f = torch.tensor(st.nodal_loads, device="cuda")
    print("270 x 270", flush=True)
    u = plan.solve(f)
    info = plan.direct_info()
    assert info["taken"] is False and info["max_front"] > 2300 and info["begun"] == info["factorisations"] == 0, info
    assert plan.last_info["levels"] > 0 and plan.last_info["converged"] == 1
    r = plan.spmv(u) - f
    r[torch.as_tensor(st.known_id.astype(np.int64), device="cuda")] = 0.0
    assert float(torch.linalg.norm(r) / torch.linalg.norm(f)) < 1e-6
