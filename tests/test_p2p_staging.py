"""The U list stages its sources through windows of 64 leaves and chunks of 512 points: trees whose
leaves hold one or a few points (more than 64 leaves to a chunk), exactly the chunk's or more than
a block's points, and duplicated points, against the direct sum.  A source left out, repeated or
moved changes its neighbours' values by far more than the expansions' error at m = 10."""
import numpy as np
import pytest

import oracle as O
import pvfmm_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kernel,n,max_pts", [
    ("laplace_poten", 600, 1), ("laplace_grad", 900, 3), ("stokes_vel", 500, 2),
    ("laplace_poten", 512, 512), ("laplace_grad", 513, 600), ("laplace_grad", 3000, 700), ("stokes_vel", 1500, 400),
])
def test_ulist_staging_matches_direct_sum(gpu, kernel, n, max_pts, prec):
    rng = np.random.default_rng(n + max_pts)
    # duplicated points only where a leaf holds them: they would split a tree of smaller leaves
    # down to the depth limit
    dup = 5 if max_pts >= 5 else 1
    x = np.concatenate([rng.random((n - n // 4, 3)), 0.7 + 0.01 * rng.random((n // 4 - dup, 3)), np.full((dup, 3), 0.31)])
    k0, _ = P.kernel_dims(kernel)
    q = rng.standard_normal(k0 * n)
    u = P.PtFMMTree(x, x, max_pts).setup(P.PtFMM(kernel, 10 if k0 == 1 else 8, prec)).evaluate(q)
    ref = O.direct(kernel, x, q, x).ravel()
    # 2-norm and largest difference, relative to the norm and the root mean square: the accuracy of
    # these orders (1e-9 at m = 10, 1e-5 for Stokes at m = 8) with a margin, FP32 rounding for mixed
    e = float(np.linalg.norm(u - ref) / np.linalg.norm(ref))
    worst = float(np.max(np.abs(u - ref)) / np.sqrt(np.mean(ref ** 2)))
    assert e < 1e-4 and worst < 1e-3, (e, worst)
