"""The separate PP and NN kernels against the oracle: rows of one to a few
columns, sectors that are no multiple of the 16-row PP or 8-row NN tiles,
neutron rows on both sides of the 2,048 columns FP64 stages at a time, and
accumulation onto an earlier y."""
import numpy as np
import pytest

from bigstickpublick_amd.inputs import small_case
from golden_cases import paths
from oracle_api import Oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("space,Z,N,jz2", [("pf", 3, 1, 0), ("pf", 4, 1, 5), ("sd", 5, 3, 0), ("pf", 2, 4, 0),
                                           ("pf", 2, 6, 0), ("pf", 1, 6, 1)])
def test_like_kernels(space, Z, N, jz2, tmp_path):
    from bigstickpublick_amd import System
    from bigstickpublick_amd.inputs import write_case
    case = small_case(space, Z, N, jz2, seed=31)
    write_case(case, str(tmp_path))
    files = paths(case, str(tmp_path))
    s = System(*files, Z, N, jz2, upload=True)
    o = Oracle(*files, Z, N, jz2)
    assert s.dim == o.dim
    _, start, sec = o.sds(0)
    # the first, the last and some rows of every proton sector
    rows = np.unique(np.concatenate([np.nonzero(sec == q)[0][[0, -1]] for q in np.unique(sec)] +
                                    [np.linspace(0, len(sec) - 1, 12).astype(int)]))
    stop = np.append(start[1:], s.dim)
    states = np.concatenate([np.arange(start[r], stop[r]) for r in rows])
    rng = np.random.default_rng(6)
    x = rng.standard_normal(s.dim)
    y0 = rng.standard_normal(s.dim)
    want = o.apply_rows(x, rows)[states]
    scale = np.abs(want).max()
    like = [v for v, i in enumerate(s.variants()) if i[3] == 2]
    n = 0
    for dt, tol in (("f64", 1e-12), ("f32", 2e-5)):
        xd = torch.tensor(x, device="cuda", dtype=torch.float64 if dt == "f64" else torch.float32)
        for v in like:
            if not s.set_variant(dt, v):
                continue
            n += 1
            y = s.apply(xd)
            assert np.abs(y.cpu().numpy()[states] - want).max() / scale < tol, (dt, v)
            ya = torch.tensor(y0, device="cuda", dtype=xd.dtype)
            s.apply(xd, ya, accumulate=True)
            assert np.abs(ya.cpu().numpy()[states] - y0[states] - want).max() / scale < tol, (dt, v)
    assert n >= 2
