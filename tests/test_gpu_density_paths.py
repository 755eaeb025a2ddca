"""The proton-neutron density by gathers (the kernel of rows that do not fit in LDS)
against the matrix-core kernel: short, odd and long rows, few and many of them.

Both round every row's sum, at most |psi|^2, to 64 |psi|^2 / 2^62 (1.4e-17 |psi|^2) and
add some 1e5 of them; a row's sum in another order is off by some 1e-16 |psi|^2: 1e-12
|psi|^2 over all."""
import numpy as np
import pytest

from bigstickpublick_amd.inputs import small_case, write_case
from golden_cases import paths

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("space,Z,N,jz2", [("sd", 1, 1, 0), ("sd", 2, 3, 1), ("pf", 3, 1, 0), ("sd", 5, 6, 1), ("pf", 2, 5, 1),
                                           ("pf", 1, 8, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_density_gather(space, Z, N, jz2, dtype, tmp_path):
    from bigstickpublick_amd import System
    case = small_case(space, Z, N, jz2, seed=67)
    write_case(case, str(tmp_path))
    s = System(*paths(case, str(tmp_path)), Z, N, jz2, upload=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    psi = torch.randn(s.dim, generator=g, device="cuda", dtype=dtype)
    tiles = s.density(psi)
    s.set_density_gather(True)
    lists = s.density(psi)
    for a, b in zip(tiles[:3], lists[:3]):
        assert np.abs(a - b).max() <= 1e-12 * tiles[3]
    assert np.abs(lists[2]).max() > 1e-3 * tiles[3]
    again = s.density(psi)
    assert all(np.array_equal(a, b) for a, b in zip(lists[:3], again[:3]))
    s.set_density_gather(False)
    back = s.density(psi)
    assert all(np.array_equal(a, b) for a, b in zip(tiles[:3], back[:3]))
    s.close()
