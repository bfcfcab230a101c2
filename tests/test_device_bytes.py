"""device_bytes of a tree: its own buffers and the operators that trees of one PtFMM share, the
transposed ones from the first adjoint evaluation on, whichever tree had it."""
import numpy as np
import pytest

import pvfmm_amd as P

pytestmark = pytest.mark.gpu


def test_device_bytes_hold_the_operators_in_use(gpu):
    rng = np.random.default_rng(2)
    m, n = 10, 400
    K = 6 * (m - 1) ** 2 + 2  # equivalent densities of a box
    fmm = P.PtFMM("laplace_poten", m, "mixed")
    xs = [rng.random((n, 3)) for _ in range(2)]
    trees = [P.PtFMMTree(x, x, 40).setup(fmm) for x in xs]
    before = [t.stats()["device_bytes"] for t in trees]
    trees[0].evaluate_adjoint(rng.standard_normal(n))
    after = [t.stats()["device_bytes"] for t in trees]
    transposed = 4 * (2 * 8 * K * K)  # U2U and D2D alone, the largest of them
    assert after[0] - before[0] > transposed  # the plan's own adjoint buffers are a tenth of that
    assert after[1] - before[1] > transposed
    again = P.PtFMMTree(xs[1], xs[1], 40).setup(fmm)
    assert again.stats()["device_bytes"] == after[1]
