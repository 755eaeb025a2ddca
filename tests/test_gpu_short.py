"""The short-row kernel against the oracle, every shape: rows of one column, of
fewer and of more columns than a wave and on both sides of a chunk's end, one to
nine chunks, sectors that are no multiple of a tile's rows, jumps that take more
than one pass through LDS, single-particle energies, accumulation."""
import numpy as np
import pytest

from bigstickpublick_amd.inputs import small_case
from golden_cases import paths
from oracle_api import Oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("space,Z,N,jz2", [("sd", 1, 0, 1), ("sd", 2, 1, 1), ("sd", 1, 6, 1), ("sd", 3, 4, 5), ("sd", 5, 6, 1),
                                           ("sd", 11, 6, 3), ("pf", 3, 2, 1), ("pf", 1, 3, 0), ("pf", 2, 17, 1), ("pf", 5, 2, 1), ("pf", 2, 4, 0),
                                           ("pf", 3, 4, 3), ("pf", 1, 16, 1)])
def test_short_rows(space, Z, N, jz2, tmp_path):
    from bigstickpublick_amd import System
    from bigstickpublick_amd.inputs import write_case
    case = small_case(space, Z, N, jz2, seed=37)
    write_case(case, str(tmp_path))
    files = paths(case, str(tmp_path))
    s = System(*files, Z, N, jz2, upload=True)
    o = Oracle(*files, Z, N, jz2)
    assert s.dim == o.dim
    _, start, sec = o.sds(0)
    # the first, the last and some rows of every proton sector
    rows = np.unique(np.concatenate([np.nonzero(sec == q)[0][[0, -1]] for q in np.unique(sec)] +
                                    [np.linspace(0, len(sec) - 1, 40).astype(int)]))
    stop = np.append(start[1:], s.dim)
    states = np.concatenate([np.arange(start[r], stop[r]) for r in rows])
    rng = np.random.default_rng(8)
    x = rng.standard_normal(s.dim)
    y0 = rng.standard_normal(s.dim)
    want = o.apply_rows(x, rows)[states]
    scale = np.abs(want).max()
    info = s.variants()
    many = (space, Z) == ("pf", 5)  # many rows: the four-row shapes only
    for dt, tol in (("f64", 1e-12), ("f32", 2e-5)):
        xd = torch.tensor(x, device="cuda", dtype=torch.float64 if dt == "f64" else torch.float32)
        s.set_variant(dt, info.index((1, 2, 0, 0)))
        tiles = s.apply(xd)
        ran = {3: 0, 4: 0, 5: 0}
        for v, i in enumerate(info):
            if i[3] < 3 or not s.set_variant(dt, v):
                continue
            ran[i[3]] += 1
            y = s.apply(xd)
            assert np.abs(y.cpu().numpy()[states] - want).max() / scale < tol, (dt, v)
            if i[3] == 4:  # the order of the tile kernel's one-row, two-jump shape
                assert torch.equal(y, tiles), (dt, v)
            ya = torch.tensor(y0, device="cuda", dtype=xd.dtype)
            s.apply(xd, ya, accumulate=True)
            assert np.abs(ya.cpu().numpy()[states] - y0[states] - want).max() / scale < tol, (dt, v)
        # sums shared by waves, in FP32 on bases of some size; in order, FP32 and rows of
        # up to 256 columns; the PN part alone, from 129 columns on
        row = (stop - start).max()
        shared = (2 if many else 5) if dt == "f64" or s.dim >= 65536 else 0
        alone = (2 if many else 4) if shared and row > 128 else 0
        assert ran == {3: shared, 4: 0 if many or dt == "f64" or row > 256 else 2, 5: alone}, (dt, ran)
