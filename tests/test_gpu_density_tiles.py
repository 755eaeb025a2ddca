"""The gradient pass where its proton-neutron tiles have remainders: classes
with more than 16 proton jumps into a row, operator classes and neutron rows
that are no multiple of 16, rows of one column.  H is linear in its
parameters, so sum_p theta_p dE/dtheta_p = <psi|H|psi> / <psi|psi>."""
import numpy as np
import pytest

from bigstickpublick_amd.inputs import small_case, write_case
from golden_cases import paths

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("space,Z,N,jz2", [("pf", 6, 2, 0), ("sd", 6, 5, 1), ("pf", 3, 1, 0), ("pf", 2, 4, 4)])
def test_gradient_sum(space, Z, N, jz2, dtype, tmp_path):
    from bigstickpublick_amd import System
    case = small_case(space, Z, N, jz2, seed=61)
    write_case(case, str(tmp_path))
    s = System(*paths(case, str(tmp_path)), Z, N, jz2, upload=True)
    it = case.interaction
    theta = np.array(list(it.spe) + [t[6] for t in it.tbmes])
    x = torch.randn(s.dim, generator=torch.Generator("cuda").manual_seed(9), device="cuda", dtype=torch.float64)
    if dtype == "f32":
        x = x.float()
    g = s.gradient(x)
    xd = x.double()
    want = (xd @ s.apply(xd) / (xd @ xd)).item()
    # the elements are rounded to FP32 (6e-8 each) where the parameters are not
    assert abs(float(g @ theta) - want) < 2e-7 * np.abs(g * theta).sum()
