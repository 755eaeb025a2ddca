"""Variant 0's two multi-vector kernels, one staged proton row a workgroup (forced) and
one wave a state (which the timing of the first use takes on few or short rows): the same
bits, on spaces where either is the faster."""
import pytest

from bigstickpublick_amd.inputs import small_case, write_case
from golden_cases import paths

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("space,Z,N,jz2,K", [("pf", 1, 4, 5, 34), ("sd", 1, 6, 1, 12), ("pf", 5, 1, 4, 3), ("sd", 5, 6, 1, 5),
                                             ("pf", 3, 3, 0, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_per_state_and_lanes(space, Z, N, jz2, K, dtype, tmp_path):
    from bigstickpublick_amd import System
    case = small_case(space, Z, N, jz2, seed=19)
    write_case(case, str(tmp_path))
    dt = "f32" if dtype == torch.float32 else "f64"

    def run(v):
        s = System(*paths(case, str(tmp_path)), Z, N, jz2, upload=True)
        assert v is None or s.set_block_variant(dt, K, v)
        g = torch.Generator(device="cuda").manual_seed(4)
        x = torch.randn((s.dim, K), generator=g, device="cuda", dtype=dtype)
        y = s.apply_block(x).clone()
        s.close()
        return y

    assert torch.equal(run(None), run(0))
