"""The SIMP shell batch (100x100 MITC-4, strongly heterogeneous: E = rho^3 * 30 GPa) on the
default route, the direct solve: compliance, displacements, shape and density gradients
against the FP64 oracle's fixture, with the bounds that the iterative routes are held to, and
invariants for every design."""
import json
import os

import numpy as np
import pytest

from jaxsso_amd import workloads as wl
from jaxsso_amd.batch import StructureBatch

pytestmark = pytest.mark.gpu

FIXTURE = os.path.join(os.path.dirname(__file__), "golden", "simp100_oracle.json")


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_simp_batch_by_the_direct_solve_vs_oracle(precision):
    with open(FIXTURE) as fh:
        fx = {r["design"]: r for r in json.load(fh)["designs"]}
    designs = [wl.simp_shell(d) for d in range(4)]
    b = StructureBatch(designs)
    print(f"simp direct {precision}", flush=True)
    C, (dc, _, dq) = b.compliance_and_gradient(precision=precision, tol=1e-10)
    info, direct = b.plan.last_info, b.plan.direct_info()
    assert info["converged"] == info["n_systems"] == 4 and info["levels"] == 0, info
    assert direct["taken"] and direct["begun"] == direct["finished"] == 1 and direct["max_front"] > 800, direct
    C, u = C.cpu().numpy()[:, 0], b.u.cpu().numpy().ravel()
    dcs, dqn = b.split_nodes(dc.cpu().numpy().reshape(-1, 3)), dq.cpu().numpy().reshape(-1, 5)
    assert {0, 1} <= set(fx)
    for d, st in enumerate(designs):
        dqd = dqn[b.quad_off[d]:b.quad_off[d + 1]]
        # K is linear in E, and a rigid translation of all nodes changes no element
        assert abs(np.sum(st.prop_quads[:, 1] * dqd[:, 1]) + C[d]) / C[d] < 1e-9
        assert np.all(np.abs(dcs[d].sum(0)) <= 1e-10 * np.abs(dcs[d]).sum(0))
        if d not in fx:
            continue
        r, o = fx[d], 6 * int(b.node_off[d])
        drho = dqd[:, 1] * 3.0 * st.rho ** 2 * 30e9
        assert abs(C[d] - r["C"]) / r["C"] < 1e-9
        assert rel(u[o:o + st.ndof][r["u_index"]], r["u"]) < 1e-8
        assert rel(dcs[d][r["dz_node"], 2], r["dz"]) < 1e-8
        assert rel(drho[r["drho_elem"]], r["drho"]) < 1e-8
        assert abs(np.linalg.norm(drho) - r["norm_drho"]) / r["norm_drho"] < 1e-8
        assert abs(np.linalg.norm(dcs[d][st.design_nodes, 2]) - r["norm_dz_free"]) / r["norm_dz_free"] < 1e-8
