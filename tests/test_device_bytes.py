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


def test_spectra_of_several_vectors_are_bounded(gpu):
    """A pass takes fewer vectors where the spectra of all would be more than 2 GiB, with the results of
    the vectors alone (to the rounding of the translations, whose K splits depend on the rows)."""
    import torch

    rng = np.random.default_rng(3)
    n, m, nv = 30000, 8, 8
    x = rng.random((n, 3))
    fmm = P.PtFMM("stokes_vel", m, "fp64")
    one, several = P.PtFMMTree(x, x, 100).setup(fmm), P.PtFMMTree(x, x, 100).setup(fmm, n_vec_max=nv)
    s = several.stats()
    spectra = 8 * 48 * m * (2 * m - 1) ** 2 * (s["v_src_slots"] + s["v_trg_slots"])  # of a vector
    assert nv * spectra > 2**32
    K = 3 * (6 * (m - 1) ** 2 + 2)
    rows = 3 * s["n_nodes"] + 2 * max(s["s2m_rows"], s["l2t_rows"]) + s["l2t_rows"]
    own = 8 * (6 * n + K * rows)  # densities, outputs and expansions of a vector
    work = 8 * 2**25  # partial products of the translations
    assert s["device_bytes"] - one.stats()["device_bytes"] < 1.02 * (nv - 1) * own + work + 2**31
    q = torch.tensor(rng.standard_normal((nv, 3 * n)), device="cuda:0")
    for got, ref in ((several.evaluate_device(q), [one.evaluate_device(v) for v in q]),
                     (several.evaluate_adjoint_device(q), [one.evaluate_adjoint_device(v) for v in q])):
        for v in range(nv):
            e = float((got[v] - ref[v]).norm() / ref[v].norm())
            # FP64 Stokes at m = 8 amplifies rounding up to 1e-5 of the result
            assert e < 1e-4, (v, e)
