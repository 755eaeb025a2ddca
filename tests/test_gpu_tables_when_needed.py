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


def test_single_vector_tables(tmp_path):
    s = _system("pf", 3, 5, 0, tmp_path)  # some 16 MiB of tables with FP32 values, 18 of FP64 values
    x = {d: torch.ones(s.dim, device="cuda", dtype=d) for d in (torch.float32, torch.float64)}
    y = {d: torch.empty_like(v) for d, v in x.items()}
    for d in x:
        s.gradient(x[d])
    s.lanczos(1, 10, dtype="f32", polish=False)
    grown = []
    for d in x:
        before = _used()
        s.apply(x[d], y[d])
        grown.append(_used() - before)
    assert min(grown) >= 8 << 20
    before = _used()
    for d in x:
        s.apply(x[d], y[d])
    assert abs(_used() - before) < 4 << 20
    s.close()


@pytest.mark.parametrize("space,Z,N,jz2", [("sd", 4, 4, 0), ("pf", 3, 4, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_first_apply_under_capture(space, Z, N, jz2, dtype, tmp_path):
    """Nothing is built under capture: the largest tile runs, now and at every replay."""
    s = _system(space, Z, N, jz2, tmp_path)
    s.upload()
    x = torch.randn(s.dim, device="cuda", dtype=dtype)
    y = torch.zeros_like(x)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        s.apply(x, y)
    eager = s.apply(x, torch.empty_like(x))  # builds the tables
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert (y - eager).abs().max() <= (2e-5 if dtype == torch.float32 else 1e-12) * eager.abs().max()
        first = y.clone() if _ == 0 else first
        assert torch.equal(y, first)
        assert torch.equal(s.apply(x, torch.empty_like(x)), eager)
    dt = "f32" if dtype == torch.float32 else "f64"
    assert s.set_variant(dt, s.variants().index((4, 4, 1, 0)))
    assert torch.equal(s.apply(x, torch.empty_like(x)), first)
    s.close()
