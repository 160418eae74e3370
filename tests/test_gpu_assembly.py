"""K exported by the assembly into the caller's buffer: 16- and 8-byte aligned buffers and
the plan's own copy hold the same bits, at block counts around the kernels' 128 blocks and
64 nodes a workgroup, at nodes with many members, and on a plan without elements."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from jaxsso_amd import _native as nat
from jaxsso_amd import workloads as wl
from jaxsso_amd.plan import FEPlan
from oracle import system
from test_gpu_direct import ribbed, spokes

pytestmark = pytest.mark.gpu

CASES = {"frames": lambda: wl.notebook_frames(3, 2), "quad3": lambda: wl.shell_pinned_edges(3, 1.0, 0.2),
         "quad7": lambda: wl.shell_pinned_edges(7, 2.0, 0.4), "quad9": lambda: wl.shell_pinned_edges(9, 2.0, 0.4),
         "grid5": lambda: wl.gridshell(5), "ribbed": ribbed, "spokes": spokes}


@pytest.mark.parametrize("case", sorted(CASES))
def test_exported_K_at_either_alignment(case):
    st = CASES[case]()
    print(f"assembly {case}: {st.n_node} nodes", flush=True)
    plan = FEPlan([0, st.n_node], st.cnct_beamcols, st.cnct_quads, st.known_id)
    crds = torch.tensor(st.crds, device="cuda")
    pb, pq = torch.tensor(st.prop_beamcols, device="cuda"), torch.tensor(st.prop_quads, device="cuda")
    K = plan.assemble(crds, pb, pq, export_K=True)
    buf = torch.full((plan.nnzb * 36 + 2,), 7.0, dtype=torch.float64, device="cuda")
    odd = buf[1:-1]
    nat.check(nat.lib().jsso_assemble(plan._h, nat.ptr(crds), nat.ptr(pb) if len(pb) else None,
                                      nat.ptr(pq) if len(pq) else None, nat.ptr(odd), nat.stream_ptr()))
    assert torch.equal(odd, K.reshape(-1)) and buf[0] == 7.0 and buf[-1] == 7.0
    rowptr, colind = plan.pattern()
    ref = system.assemble_K(st.crds, st.cnct_beamcols, st.prop_beamcols, st.cnct_quads, st.prop_quads)
    rows = np.repeat(np.arange(st.n_node), np.diff(rowptr))
    got = K.cpu().numpy()
    dense = np.zeros((6 * st.n_node, 6 * st.n_node))
    for b, (i, j) in enumerate(zip(rows, colind)):
        dense[6 * i:6 * i + 6, 6 * j:6 * j + 6] = got[b]
    # sums of up to 70 element entries of one size: rounding, 1e-13 of the largest
    assert np.abs(dense - ref.toarray()).max() < 1e-13 * np.abs(dense).max()
    x = torch.randn(st.ndof, dtype=torch.float64, device="cuda")
    assert torch.equal(plan.spmv(x), plan.spmv(x, K=K))   # the plan's own copy, filled on demand


def test_plan_without_elements():
    plan = FEPlan([0, 3], np.zeros((0, 2), np.int32), np.zeros((0, 4), np.int32), np.arange(18))
    K = plan.assemble(torch.zeros(3, 3, dtype=torch.float64), None, None, export_K=True)
    assert K.shape == (3, 6, 6) and not K.any()
