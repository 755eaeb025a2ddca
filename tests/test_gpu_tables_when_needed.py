"""Tables that only some kernels read are built when one of those is first wanted: device
memory in use before and after."""
import pytest

from bigstickpublick_amd.inputs import small_case, write_case
from golden_cases import paths

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _system(space, Z, N, jz2, d):
    from bigstickpublick_amd import System
    case = small_case(space, Z, N, jz2, seed=23)
    write_case(case, str(d))
    return System(*paths(case, str(d)), Z, N, jz2, upload=True)


def _used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_k_vector_lists(tmp_path):
    s = _system("pf", 3, 5, 0, tmp_path)  # 1.2 million neutron one-body entries of 8 bytes
    before = []
    for K, dtype in ((64, torch.float64), (3, torch.float32)):  # rows of 64 do not fit in LDS
        x = torch.ones((s.dim, K), device="cuda", dtype=dtype)
        y = torch.empty_like(x)
        before.append(_used())
        s.apply_block(x, y)
    assert _used() - before[1] >= 8 << 20
    assert torch.equal(y[:, 0], y[:, 2])
    s.close()
