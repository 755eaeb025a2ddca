"""FP32 solves keep one order of a column's sum per space: the bits of the shape the
space's sizes name, in every System and whatever variant H x alone takes."""
import numpy as np
import pytest

from bigstickpublick_amd.inputs import small_case
from golden_cases import paths

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# (rows, staged) of the order: two jumps of a row, R2 G4, R2 G2, the row kernel
@pytest.mark.parametrize("space,Z,N,jz2,shape", [("sd", 4, 4, 0, (1, 2)), ("sd", 5, 6, 1, (2, 4)), ("pf", 3, 3, 0, (2, 2)),
                                                 ("pf", 3, 4, 1, (2, 2)), ("pf", 2, 5, 1, (1, 2)), ("pf", 4, 2, 0, (1, 0)),
                                                 ("pf", 1, 6, 1, (1, 0))])
def test_fp32_solve_order(space, Z, N, jz2, shape, tmp_path):
    from bigstickpublick_amd import System
    from bigstickpublick_amd.inputs import write_case
    case = small_case(space, Z, N, jz2, seed=41)
    write_case(case, str(tmp_path))
    files = paths(case, str(tmp_path))

    def solve(how):
        s = System(*files, Z, N, jz2, upload=True)
        how(s)
        r = s.lanczos(3, 25, dtype="f32", want_vectors=True, polish=False)
        return r.alpha, r.beta, r.evecs

    def named(s):
        assert s.set_variant("f32", [i[:2] for i in s.variants()].index(shape))

    want = solve(named)
    for how in (lambda s: s.autotune("f32"), lambda s: s.autotune("f32")):
        got = solve(how)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert torch.equal(got[2], want[2])
    # until tuned: the order of the largest tile
    if shape != (1, 0):
        largest = solve(lambda s: s.set_variant("f32", [i[:2] for i in s.variants()].index((4, 4))))
        assert torch.equal(solve(lambda s: None)[2], largest[2])


# K vectors: the order of the fastest among the per-state kernel (variant 0) and the
# tile kernels (one staged jump 1, two 3), though the kernel that shares variant 0's bits
# may be faster than the one, or slower than the other
@pytest.mark.parametrize("what,space,Z,N,jz2,K,orders", [("block", "sd", 4, 10, 4, 8, (1, 3)), ("batch", "sd", 4, 10, 4, 8, (1, 3)),
                                                         ("batch", "pf", 4, 1, 5, 4, (0,)), ("batch", "sd", 6, 5, 1, 3, (0,))])
def test_fp32_k_vector_solve_order(what, space, Z, N, jz2, K, orders, tmp_path):
    from bigstickpublick_amd import Batch, System
    from bigstickpublick_amd.inputs import write_case
    files = []
    for k in range(K if what == "batch" else 1):
        case = small_case(space, Z, N, jz2, seed=50 + k)
        case.name += "_%d" % k
        write_case(case, str(tmp_path))
        files.append(paths(case, str(tmp_path)))

    def solve(v):
        if what == "batch":
            b = Batch(files[0][0], [f[1] for f in files], Z, N, jz2)
            assert v is None or b.set_variant("f32", v)
            r = b.lanczos(2, 20, dtype="f32", want_vectors=True, polish=False)
        else:
            b = System(*files[0], Z, N, jz2, upload=True)
            assert v is None or b.set_block_variant("f32", K, v)
            r = b.block_lanczos(4, 6 * K, K, dtype="f32", want_vectors=True, polish=False)
        vec = r.evecs.clone()
        b.close()
        return vec

    got = solve(None)
    assert any(torch.equal(got, solve(v)) for v in orders)
