"""The direct solve (multifrontal Cholesky, the default of a plan whose caller has not
chosen a preconditioner) against the oracle, at the sizes where its kernels change:
single-front structures, one-workgroup fronts of every padding, fronts in panels,
several components, both element types, 1 to 4 load cases, uneven batches."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from jaxsso_amd import _native as nat
from jaxsso_amd import workloads as wl
from jaxsso_amd.batch import StructureBatch
from jaxsso_amd.plan import FEPlan
from oracle import solve as osolve
from oracle import system

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - b) / max(np.linalg.norm(b), 1e-300))


def oracle_u(st, f):
    K = system.assemble_K(st.crds, st.cnct_beamcols, st.prop_beamcols, st.cnct_quads, st.prop_quads)
    return osolve.solve_reduced(K, st.known_id, f)


def two_parts():
    """Two shells that share nothing, as one structure."""
    a, b = wl.shell_pinned_edges(9, 4.0, 0.6, design=1), wl.shell_pinned_edges(5, 3.0, 0.5, design=2)
    n = a.n_node
    return wl.Structure(np.concatenate([a.crds, b.crds]), np.zeros((0, 2), np.int32), np.zeros((0, 6)),
                        np.concatenate([a.cnct_quads, b.cnct_quads + n]).astype(np.int32),
                        np.concatenate([a.prop_quads, b.prop_quads]),
                        np.concatenate([a.known_id, b.known_id + 6 * n]).astype(np.int32),
                        np.concatenate([a.nodal_loads, b.nodal_loads]), name="two parts")


def spokes(n=70):
    """A hub with n beams to pinned nodes: one node with n neighbours."""
    t = 2 * np.pi * (np.arange(n) + 0.3) / n
    crds = np.concatenate([[[0.0, 0.0, 1.0]], np.stack([3 * np.cos(t), 3 * np.sin(t), 0 * t], 1)])
    cnct = np.stack([np.zeros(n, int), 1 + np.arange(n)], 1).astype(np.int32)
    loads = np.zeros(6 * (n + 1))
    loads[2] = -1000.0
    return wl.Structure(crds, cnct, wl._beam_props(n), np.zeros((0, 4), np.int32), np.zeros((0, 5)),
                        wl._support_ids(1 + np.arange(n), [1] * 6), loads, name="spokes")


def ribbed(n=23):
    st = wl.shell_pinned_edges(n, 5.0, 0.8, design=4)
    st.crds[st.design_nodes, 2] += np.random.default_rng(2).normal(0.0, 0.01, len(st.design_nodes))
    node = np.arange((n + 1) ** 2).reshape(n + 1, n + 1)
    rows = node[4:n:5]
    st.cnct_beamcols = np.stack([rows[:, :-1].ravel(), rows[:, 1:].ravel()], 1).astype(np.int32)
    st.prop_beamcols = wl._beam_props(len(st.cnct_beamcols))
    return st


SINGLE = {"two_nodes": lambda: wl.notebook_frames(3, 2), "quad2": lambda: wl.shell_pinned_edges(2, 1.0, 0.2),
          "quad3": lambda: wl.shell_pinned_edges(3, 1.0, 0.2), "quad7": lambda: wl.shell_pinned_edges(7, 2.0, 0.4),
          "quad16": lambda: wl.shell_pinned_edges(16, 4.0, 0.6), "quad33": lambda: wl.shell_pinned_edges(33, 8.0, 1.2),
          "quad70": lambda: wl.shell_pinned_edges(70, 12.0, 2.0), "grid5": lambda: wl.gridshell(5),
          "grid19": lambda: wl.gridshell(19), "two_parts": two_parts, "spokes": spokes, "ribbed": ribbed}


@pytest.mark.parametrize("case", sorted(SINGLE))
def test_direct_solve_matches_oracle(case):
    st = SINGLE[case]()
    print(f"direct {case}: {st.n_node} nodes", flush=True)
    plan = FEPlan([0, st.n_node], st.cnct_beamcols, st.cnct_quads, st.known_id)
    plan.assemble(torch.tensor(st.crds), torch.tensor(st.prop_beamcols), torch.tensor(st.prop_quads))
    u = plan.solve(torch.tensor(st.nodal_loads)).cpu().numpy()
    info = plan.last_info
    # at most a few refinement steps: the AMG's iterations are counted in tens
    assert info["converged"] == 1 and info["levels"] == 0 and info["iterations"] <= 6, info
    ur = oracle_u(st, st.nodal_loads)
    assert rel(u, ur) < 1e-8, info
    assert np.all(u[st.known_id] == 0.0)
    if case == "spokes":
        return   # (the AMG cannot coarsen a hub whose neighbours are all held: its CG does not start there)
    # the same plan with the preconditioner chosen: the iterative route, the same u
    v = plan.solve(torch.tensor(st.nodal_loads), preconditioner="amg", tol=1e-11).cpu().numpy()
    assert plan.last_info["levels"] > 0 and rel(u, v) < 1e-8


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 4])
def test_direct_batch_of_uneven_designs(precision, nrhs):
    """Structures of different and of equal patterns (the same mesh twice shares one
    analysis), several load cases, a second assembly on the plan, and a structure
    without load."""
    designs = [wl.cfg1(0), wl.gridshell(9, noise=0.1, cfg=3, design=5, half_span_cases=True),
               wl.shell_pinned_edges(12, 8.0, 1.0, design=2), wl.cfg1(1)]
    designs[2].nodal_loads[:] = 0.0
    b = StructureBatch(designs, n_cases=nrhs)
    print(f"direct batch {precision} nrhs {nrhs}", flush=True)
    for scale in (1.0, 1.3):
        b.prop_quad[:, 0] *= scale
        u = b.solve(precision=precision).cpu().numpy().reshape(-1, nrhs)
        info = b.plan.last_info
        assert info["converged"] == info["n_systems"] == 4 * nrhs and info["levels"] == 0, info
        pq = b.prop_quad.cpu().numpy()
        for i, st in enumerate(designs):
            st.prop_quads = pq[b.quad_off[i]:b.quad_off[i + 1]]
            o = 6 * int(b.node_off[i])
            for c, f in enumerate(st.load_cases()[:nrhs]):
                got = u[o:o + st.ndof, c]
                assert rel(got, oracle_u(st, f)) < 1e-8 if f.any() else not got.any(), (scale, i, c, info)


def test_direct_solve_repeats_itself_and_hands_over_what_it_does_not_take():
    """Two solves of one assembly agree bit for bit; eight load cases and a plan asked to
    keep its AMG hierarchy take the iterative route."""
    b = StructureBatch([wl.cfg1(0), wl.shell_pinned_edges(12, 8.0, 1.0, design=2)])
    u0 = b.solve().clone()
    assert b.plan.last_info["levels"] == 0
    assert torch.equal(u0, b.solve()) and torch.equal(u0, b.solve(assemble=False))
    f8 = b.f.reshape(-1, 1) * torch.arange(1, 9, device=b.f.device, dtype=torch.float64)
    u8 = b.plan.solve(f8.contiguous())
    assert b.plan.last_info["levels"] > 0 and rel(u8[:, 0].cpu().numpy(), u0.cpu().numpy()) < 1e-8
    b.plan.amg_reuse(2)
    u1 = b.solve()
    assert b.plan.last_info["levels"] > 0 and rel(u1.cpu().numpy(), u0.cpu().numpy()) < 1e-8


def orthotropic(n, kx, ky):
    st = wl.shell_pinned_edges(n, 0.3 * n, 0.05 * n, design=3)
    st.prop_quads[:, 3], st.prop_quads[:, 4] = kx, ky
    return st


@pytest.mark.parametrize("nrhs", [1, 3])
@pytest.mark.parametrize("kx,ky", [(1.2, 0.8), (2.0, 0.5), (0.3, 3.0)])
def test_orthotropic_batch_by_refinement_with_the_symmetric_part(kx, ky, nrhs):
    """K and K^T solves of shells of two sizes (several load cases, a structure without
    load) against the oracle's refined direct solves; the dense LU agrees."""
    designs = [orthotropic(6, kx, ky), orthotropic(17, kx, ky), orthotropic(9, kx, ky)]
    designs[2].nodal_loads[:] = 0.0
    rng = np.random.default_rng(5)
    for st in designs[:2]:
        st.extra_loads = [st.nodal_loads * rng.uniform(0.0, 2.0, st.ndof) for _ in range(nrhs - 1)]
    b = StructureBatch(designs, n_cases=nrhs)
    b.assemble()
    assert not b.plan.symmetric()
    f = b.f[:, 0].contiguous() if nrhs == 1 else b.f
    got = {t: b.plan.solve(f, transpose=t) for t in (False, True)}
    info = b.plan.last_info
    assert info["converged"] == info["n_systems"] == 3 * nrhs, info
    b.plan.nonsymmetric_route(1)
    for t in (False, True):
        dense = b.plan.solve(f, transpose=t)
        assert b.plan.last_info["iterations"] == 0
        assert rel(got[t].cpu().numpy(), dense.cpu().numpy()) < 1e-9
        u = got[t].cpu().numpy().reshape(-1, nrhs)
        for i, st in enumerate(designs):
            K = system.assemble_K(st.crds, st.cnct_beamcols, st.prop_beamcols, st.cnct_quads, st.prop_quads)
            o = 6 * int(b.node_off[i])
            for c, fc in enumerate(st.load_cases()[:nrhs]):
                v = u[o:o + st.ndof, c]
                ref = osolve.solve_reduced(K.T.tocsr() if t else K, st.known_id, fc)
                assert rel(v, ref) < 1e-9 if fc.any() else not v.any(), (t, i, c)


@pytest.mark.parametrize("m", [1, 4, 5])
def test_dense_solve_of_the_plans_own_assembly(m):
    """plan.dense_solve without K values (1 to 4 right-hand sides through the direct
    factorisation, more through the dense one) against the dense factorisation of the
    exported K and the oracle."""
    st = wl.notebook_barrel()
    plan = FEPlan([0, st.n_node], st.cnct_beamcols, st.cnct_quads, st.known_id)
    K = plan.assemble(torch.tensor(st.crds), None, torch.tensor(st.prop_quads), export_K=True)
    F = np.random.default_rng(3).normal(size=(st.ndof, m))
    f = torch.tensor(F[:, 0] if m == 1 else F, device="cuda")
    u, v = plan.dense_solve(f), plan.dense_solve(f, K=K)
    assert rel(u.cpu().numpy(), v.cpu().numpy()) < 1e-9
    ref = oracle_u(st, F)
    assert rel(u.cpu().numpy().reshape(-1, m), ref) < 1e-9


@pytest.mark.parametrize("copies", [1, 3, 64])
def test_fronts_in_panels_of_few_and_of_many_structures(copies):
    """40 x 40 shells, whose upper fronts go in panels: few structures (the update of a panel
    factors the next panel's block, a panel's columns are solved for in parts) and 64 of them
    (launches of their own), against the oracle."""
    designs = []
    for i in range(copies):
        st = wl.shell_pinned_edges(40, 10.0, 1.5, design=4)
        st.crds[st.design_nodes, 2] += np.random.default_rng(i).normal(0.0, 0.01, len(st.design_nodes))
        designs.append(st)
    b = StructureBatch(designs)
    print(f"direct panels x {copies}", flush=True)
    u = b.solve().cpu().numpy().ravel()
    info = b.plan.last_info
    assert info["converged"] == copies and info["levels"] == 0, info
    for i in {0, copies // 2, copies - 1}:
        o, st = 6 * int(b.node_off[i]), designs[i]
        assert rel(u[o:o + st.ndof], oracle_u(st, st.nodal_loads)) < 1e-8, (i, info)


@pytest.mark.parametrize("kinds", ["sym sym ortho sym ortho ortho", "ortho sym sym", "sym bad sym"])
def test_assemblies_that_change_kind_on_one_plan(kinds):
    """The direct solve starts before the assembly's flags are known where the last ones
    allowed it: K that is or is not symmetric, or has a diagonal block that is not positive
    definite, in any order on one plan, also with the result over the right-hand side."""
    st = orthotropic(9, 1.0, 1.0)
    plan = FEPlan([0, st.n_node], st.cnct_beamcols, st.cnct_quads, st.known_id)
    f = torch.tensor(st.nodal_loads, device="cuda")
    for kind in kinds.split():
        print(f"direct flags {kind}", flush=True)
        pq = st.prop_quads.copy()
        pq[:, 3:] = (1.5, 0.6) if kind == "ortho" else (1.0, 1.0)
        if kind == "bad":
            pq[:, 1] *= -1.0
        plan.assemble(torch.tensor(st.crds), None, torch.tensor(pq))
        if kind == "bad":
            with pytest.raises(RuntimeError):
                plan.solve(f)
            continue
        u = plan.solve(f).cpu().numpy()
        K = system.assemble_K(st.crds, st.cnct_beamcols, st.prop_beamcols, st.cnct_quads, pq)
        assert rel(u, osolve.solve_reduced(K, st.known_id, st.nodal_loads)) < 1e-8, kind
        # in place, and again with the flags unread
        plan.assemble(torch.tensor(st.crds), None, torch.tensor(pq))
        v, info = f.clone(), nat.Info()
        nat.check(nat.lib().jsso_solve(plan._h, nat.ptr(v), nat.ptr(v), 1, nat.PREC["fp64"], 1e-12, 1000,
                                       ctypes.byref(info), nat.stream_ptr()), allow_not_converged=True)
        assert rel(v.cpu().numpy(), u) < 1e-8, kind
