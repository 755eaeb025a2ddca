"""The multi-vector kernel that stages a proton row's jumps (variant 0) against
the oracle: groups of 8 to 64 lanes filled and not, odd numbers of vectors,
rows of one column to some dozens, vectors that start off a 16-byte boundary,
one Hamiltonian for all and one per vector."""
import os

import numpy as np
import pytest

from bigstickpublick_amd.inputs import small_case, write_case
from golden_cases import ensemble_fixture, paths
from oracle_api import Oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-12, "f32": 2e-5}
TYPE = {"f64": torch.float64, "f32": torch.float32}


def _off(x, dtype):
    """x on the device, one element off its allocation's start"""
    buf = torch.empty(x.size + 1, device="cuda", dtype=dtype)
    v = buf[1:].view(*x.shape)
    v.copy_(torch.tensor(x))
    return v


@pytest.mark.parametrize("space,Z,N,jz2", [("sd", 2, 3, 1), ("pf", 3, 1, 0), ("pf", 2, 2, 0), ("sd", 5, 5, 4)])
@pytest.mark.parametrize("K", [1, 3, 8, 9, 16, 17, 32, 33, 64])
def test_block_lanes(space, Z, N, jz2, K, tmp_path):
    from bigstickpublick_amd import System
    case = small_case(space, Z, N, jz2, seed=17)
    write_case(case, str(tmp_path))
    files = paths(case, str(tmp_path))
    s = System(*files, Z, N, jz2, upload=True)
    o = Oracle(*files, Z, N, jz2)
    X = np.random.default_rng(K).standard_normal((s.dim, K))
    cols = sorted({0, K // 2, K - 1})
    want = {k: o.apply(np.ascontiguousarray(X[:, k])) for k in cols}
    for dt, tol in TOL.items():
        assert s.set_block_variant(dt, K, 0)
        for xd in (torch.tensor(X, device="cuda", dtype=TYPE[dt]), _off(X, TYPE[dt])):
            y = s.apply_block(xd).cpu().numpy()
            for k in cols:
                assert np.abs(y[:, k] - want[k]).max() / np.abs(want[k]).max() < tol, (dt, k)


@pytest.mark.parametrize("K", [3, 12, 33])
def test_batch_lanes(casedir, K):
    from bigstickpublick_amd import Batch
    cases, d, fx = ensemble_fixture(casedir, K)
    b = Batch(os.path.join(d, "sd.sps"), [paths(c, d)[1] for c in cases], 4, 4, 0)
    X = np.random.default_rng(3).standard_normal((b.dim, K))
    cols = sorted({0, K // 2, K - 1})
    want = {k: Oracle(*paths(cases[k], d), 4, 4, 0).apply(np.ascontiguousarray(X[:, k])) for k in cols}
    for dt, tol in TOL.items():
        assert b.set_variant(dt, 0)
        for xd in (torch.tensor(X, device="cuda", dtype=TYPE[dt]), _off(X, TYPE[dt])):
            y = b.apply(xd).cpu().numpy()
            for k in cols:
                assert np.abs(y[:, k] - want[k]).max() / np.abs(want[k]).max() < tol, (dt, k)
    b.close()
