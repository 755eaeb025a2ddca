"""The batched tridiagonal Ritz solve against LAPACK on the coefficients of the
same run, from one step to more than a wave's 64, and up to 16 vectors."""
import numpy as np
import pytest

from bigstickpublick_amd.inputs import small_case, write_case
from golden_cases import paths

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,niter,nkeep", [(1, 1, 1), (3, 2, 2), (2, 16, 16), (5, 20, 3), (2, 70, 7)])
def test_batched_ritz(K, niter, nkeep, tmp_path):
    from bigstickpublick_amd import Batch
    files = []
    for k in range(K):
        case = small_case("sd", 2, 3, 1, seed=50 + k)
        write_case(case, str(tmp_path / str(k)))
        sps, f = paths(case, str(tmp_path / str(k)))
        files.append(f)
    b = Batch(sps, files, 2, 3, 1)
    r = b.lanczos(nkeep, niter, dtype="f64", polish=False, want_vectors=True)
    for k in range(K):
        t = np.diag(r.alpha[k]) + np.diag(r.beta[k][:niter - 1], 1) + np.diag(r.beta[k][:niter - 1], -1)
        want = np.linalg.eigvalsh(t)[:nkeep]
        # bisection stops at 1e-15 (|l| + |h|), the counts are backward stable
        assert np.abs(r.evals[k] - want).max() < 1e-13 * np.abs(t).sum(axis=1).max(), (k, r.evals[k], want)
        # orthonormal Ritz vectors of orthonormal Lanczos vectors
        x = r.evecs[:, :, k].double()
        assert (x @ x.t() - torch.eye(nkeep, device="cuda", dtype=torch.float64)).abs().max().item() < 1e-9
