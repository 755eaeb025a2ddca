"""Every Ritz vector of a plain run satisfies the Lanczos relation: with y the eigenvector
of the run's tridiagonal matrix, |H x - E x| = |beta_m y_m| and <x_p|H|x_q> = E_q on the
diagonal, zero off it.  Batched and single, FP64, and FP32 to what its rounding leaves.

The vectors are kept orthogonal to some 1e-14 (FP64), H has norm |T|; x = V y is exact to
m eps, y to eps |T| / gap, so with gaps from 1e-3 |T| on all of it agrees to some 1e-11
|T|.  FP32: vectors rounded to 6e-8, orthogonal to some 1e-6, H x to 5e-7 |T|: 1e-5 |T|."""
import numpy as np
import pytest

from bigstickpublick_amd.inputs import small_case, write_case
from golden_cases import paths

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-11, "f32": 1e-5}


def _check(alpha, beta, evals, x, hx, tol):
    """x, hx: (nkeep, dim) FP64"""
    m, n = len(alpha), len(evals)
    t = np.diag(alpha) + np.diag(beta[:m - 1], 1) + np.diag(beta[:m - 1], -1)
    norm = np.abs(t).sum(axis=1).max()
    e, y = np.linalg.eigh(t)
    assert np.abs(e[:n] - evals).max() < tol * norm
    h = (x @ hx.t()).cpu().numpy()
    assert np.abs(h - np.diag(evals)).max() < tol * norm
    r = (hx - torch.tensor(evals, device="cuda")[:, None] * x).norm(dim=1).cpu().numpy()
    gap = np.array([np.abs(np.delete(e, q) - e[q]).min() for q in range(n)]) if m > 1 else np.full(n, norm)
    apart = gap > 1e-3 * norm
    assert apart.any()
    assert np.abs(r - np.abs(beta[m - 1] * y[m - 1, :n]))[apart].max() < tol * norm


@pytest.mark.parametrize("K,niter,nkeep", [(1, 1, 1), (3, 2, 2), (2, 16, 16), (5, 20, 3), (2, 70, 7)])
@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_batch(K, niter, nkeep, dt, tmp_path):
    from bigstickpublick_amd import Batch
    files = []
    for k in range(K):
        case = small_case("sd", 2, 3, 1, seed=50 + k)
        write_case(case, str(tmp_path / str(k)))
        sps, f = paths(case, str(tmp_path / str(k)))
        files.append(f)
    b = Batch(sps, files, 2, 3, 1)
    r = b.lanczos(nkeep, niter, dtype=dt, polish=False, want_vectors=True)
    hx = [b.apply(r.evecs[q].double().contiguous()) for q in range(nkeep)]
    for k in range(K):
        _check(r.alpha[k], r.beta[k], r.evals[k], r.evecs[:, :, k].double(), torch.stack([h[:, k] for h in hx]), TOL[dt])
    b.close()


@pytest.mark.parametrize("space,Z,N,jz2,niter,nkeep", [("sd", 2, 3, 1, 1, 1), ("sd", 5, 6, 1, 30, 5), ("pf", 3, 3, 0, 25, 3),
                                                       ("pf", 3, 4, 1, 40, 4), ("pf", 1, 6, 1, 20, 2)])
@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_single(space, Z, N, jz2, niter, nkeep, dt, tmp_path):
    from bigstickpublick_amd import System
    case = small_case(space, Z, N, jz2, seed=53)
    write_case(case, str(tmp_path))
    s = System(*paths(case, str(tmp_path)), Z, N, jz2, upload=True)
    s.autotune(dt)
    r = s.lanczos(nkeep, niter, dtype=dt, polish=False, want_vectors=True)
    x = r.evecs.double()
    _check(r.alpha, r.beta, r.evals, x, torch.stack([s.apply(x[q].contiguous()) for q in range(nkeep)]), TOL[dt])
    # polished: Rayleigh quotients of the same vectors, and their residuals
    p = s.lanczos(nkeep, niter, dtype=dt, polish=True, want_vectors=True)
    x = p.evecs.double()
    hx = torch.stack([s.apply(x[q].contiguous()) for q in range(nkeep)])
    norm = np.abs(r.alpha).max() + 2 * np.abs(r.beta).max()
    assert np.abs((x * hx).sum(1).cpu().numpy() / (x * x).sum(1).cpu().numpy() - p.evals).max() < (1e-12 if dt == "f64" else 1e-9) * norm
    assert np.abs((hx - torch.tensor(p.evals, device="cuda")[:, None] * x).norm(dim=1).cpu().numpy() - p.resid).max() < \
        (1e-11 if dt == "f64" else 1e-6) * norm
    s.close()
