"""The rounding of the mixed evaluator, against the FP64 evaluator at the FP32 pseudo-inverse cutoff on
the same tree: the same operators in 64 bits, so that the difference is the FP32 arithmetic alone.

The mean of the relative error over 60 random inputs is a steady figure (about 2% between sets of
inputs).  With the V list transformed on 2m points per axis it was 1.93e-7 (8,000 points, m = 8),
2.14e-7 (16,000, m = 8) and 2.05e-7 (16,000, m = 10), 2.04e-7 together; the grid of 2m - 1 points has to
be as accurate."""
import numpy as np
import pytest

import pvfmm_amd as P

pytestmark = pytest.mark.gpu


def test_mean_rounding_error_of_the_mixed_evaluator(gpu):
    import torch

    means = []
    for n, m in ((8000, 8), (16000, 8), (16000, 10)):
        mixed, fp64 = P.PtFMM("laplace_poten", m, "mixed"), P.PtFMM("laplace_poten", m, "fp64", pinv_cutoff=4 * 2.0**-23)
        errs = []
        for seed in range(60):
            rng = np.random.default_rng([seed, 77])
            x = rng.random((n, 3))
            q = torch.tensor(rng.standard_normal(n), device="cuda:0")
            t = P.PtFMMTree(x, x, 128)
            a = t.setup(mixed).evaluate_device(q)
            b = t.setup(fp64).evaluate_device(q)
            errs.append(float((a - b).norm() / b.norm()))
        means.append(float(np.mean(errs)))
        print(f"{n} points, m = {m}: mean relative error {means[-1]:.3e}", flush=True)
    assert np.mean(means) < 2.05e-7, means
