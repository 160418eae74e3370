"""More or fewer element-parameter values than there are parameters, for models whose
parameters are all of one element type (their values need no selection) and of both."""
import numpy as np
import pytest
import torch

import jaxsso_amd.model as Model
from jaxsso_amd.SSO_model import ElementParameter, NodeParameter, SSO_model

pytestmark = pytest.mark.gpu


def model():
    m = Model.Model()
    for j in range(4):
        for i in range(4):
            m.add_node(4 * j + i, float(i), float(j), 0.1 * i * j)
    e = 0
    for j in range(3):
        for i in range(3):
            b = 4 * j + i
            m.add_quad(e, b, b + 1, b + 5, b + 4, 0.1, 30e9, 0.3, 1.0, 1.0)
            e += 1
    for i in range(3):
        m.add_beamcol(i, 4 + i, 5 + i, 200e9, 80e9, 1e-4, 1e-4, 1e-4, 1e-2)
    for n in (0, 3, 12, 15):
        m.add_support(n, [1] * 6)
    m.add_nodal_load(5, [0.0, 0.0, -1000.0, 0.0, 0.0, 0.0])
    m.model_ready()
    return m


@pytest.mark.parametrize("types", ["quad", "beam", "both"])
def test_longer_values_are_cut_and_shorter_refused(types):
    s = SSO_model(model())
    for n in (5, 6, 9):
        s.add_nodeparameter(NodeParameter(n, 2))
    if types != "beam":
        for e in range(9):
            s.add_eleparameter(ElementParameter(e, 1, 0))
    if types != "quad":
        for e in range(3):
            s.add_eleparameter(ElementParameter(e, 0, 5))
    s.initialize_parameters_values()
    s.set_objective("strain energy")
    p = torch.tensor(s.parameter_values, device="cuda")
    C = float(s.helper_params_to_objective(p))
    longer = torch.cat([p, torch.full((4,), 7.0, dtype=p.dtype, device=p.device)]).requires_grad_(True)
    val = s.helper_params_to_objective(longer)
    (g,) = torch.autograd.grad(val, longer)
    assert float(val.detach()) == C and not g[-4:].any() and g[:-4].abs().min() > 0
    n = s.n_ele_params
    for k in (0, 1, n - 1):
        with pytest.raises(ValueError):
            s.ele_params_props(np.ones(k))
        with pytest.raises(ValueError):
            s.helper_params_to_objective(p[:3 + k])
