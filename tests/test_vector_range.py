"""The mixed evaluator on one and on 8 density vectors whose charges differ by 2^16 to 2^32 in size
within one run of V-list tiles, against the FP64 evaluator at the FP32 pseudo-inverse cutoff on the
same tree (the same operators, so that only the rounding differs).

Two clusters of 6,000 points lie far apart; the charges of one are strong, in pairs of opposite sign
0.4% of the cluster apart, so that at the other cluster its field is below the rounding of the weak
charges' own.  FP32 spectra keep their 24 bits whatever their size (2.5e-7 to 3.0e-7 at the weak
cluster when each was multiplied with its own exponent); fp16 parts of a common scale keep them only
if the second part has a scale of its own, and beyond 2^24 only if weak and strong spectra are
multiplied apart.  The bar is three times those errors."""
import numpy as np
import pytest

import pvfmm_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv", [1, 8])
@pytest.mark.parametrize("kernel,size,ratio,tol", [
    ("laplace_grad", 2.0**-9, 2.0**20, 7.5e-7),
    ("laplace_grad", 2.0**-12, 2.0**16, 7.5e-7),
    ("laplace_grad", 2.0**-12, 2.0**32, 8e-7),
    ("laplace_poten", 2.0**-12, 2.0**16, 9e-7),
])
def test_weak_cluster_far_from_a_strong_one(gpu, kernel, size, ratio, tol, nv):
    import torch

    rng = np.random.default_rng(3)
    n = 6000
    a = rng.random((n // 2, 3))
    a = np.concatenate([a, np.clip(a + 0.004 * rng.standard_normal(a.shape), 0, 1)])
    x = np.concatenate([0.125 + size * a, 0.8125 + size * rng.random((n, 3))])
    qa = ratio * rng.standard_normal((nv, n // 2))
    q = torch.tensor(np.concatenate([qa, -qa, rng.standard_normal((nv, n))], axis=1), device="cuda:0")
    t = P.PtFMMTree(x, x, 60)
    u = []
    for fmm in (P.PtFMM(kernel, 10, "mixed"), P.PtFMM(kernel, 10, "fp64", pinv_cutoff=4 * 2.0**-23)):
        t.setup(fmm, n_vec_max=nv)
        u.append(t.evaluate_device(q if nv > 1 else q[0].contiguous()).reshape(nv, 2 * n, -1)[:, n:])
    e = float((u[0] - u[1]).norm() / u[1].norm())
    print(f"{kernel}, {nv} vectors, ratio {ratio:.0f}: rel-L2 at the weak cluster {e:.2e}")
    assert e < tol, e
