"""Far-field rows with many W items are split over several blocks whose sums are added afterwards:
trees with such rows, one density vector and more than one chunk of 8, against the direct sum."""
import numpy as np
import pytest

import oracle as O
import pvfmm_amd as P
from pvfmm_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kernel,m,nv", [("laplace_poten", 10, 1), ("laplace_grad", 10, 9), ("stokes_vel", 8, 2)])
def test_split_far_rows_match_direct_sum(gpu, kernel, m, nv, prec):
    rng = np.random.default_rng(21)
    nc = 40000  # a cluster in a thin uniform cloud: coarse leaves of up to 250 points beside fine ones
    x = np.concatenate([0.3 + 0.03 * rng.standard_normal((nc, 3)), W.uniform(rng, 3000)])
    n, (k0, k1), ns = len(x), P.kernel_dims(kernel), 6 * (m - 1) ** 2 + 2
    tree = P.PtFMMTree(x, x, 250).setup(P.PtFMM(kernel, m, prec), n_vec_max=nv)
    # rows above the splitting threshold of 131072 pairs
    nodes, wl = tree.nodes(), tree.lists(12)
    cnt = nodes[:, 8]
    used = (wl >= 0) & (cnt[np.maximum(wl, 0)] > 0) & ~((nodes[np.maximum(wl, 0), 4] == 1) & (cnt[np.maximum(wl, 0)] <= ns))
    pairs = (1 + used.sum(1)) * ns * np.where(nodes[:, 4] == 1, nodes[:, 9], 0)
    assert np.any((pairs > 131072) & (used.sum(1) > 0))
    q = rng.standard_normal((nv, k0 * n))
    u = tree.evaluate(q)
    idx = np.concatenate([rng.choice(n, 200, replace=False), nc + rng.choice(3000, 800, replace=False)])
    for v in range(nv):
        ref = O.direct(kernel, x, q[v], x[idx]).ravel()
        got = u[v].reshape(n, k1)[idx].ravel()
        e = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
        # the accuracy of the orders (1e-8 at m = 10, 1e-5 for Stokes at m = 8), FP32 rounding for mixed
        assert e < (2e-4 if kernel == "stokes_vel" else 1e-6 if prec == "fp64" else 2e-5), (v, e)
