"""FP64 against the oracle on the same tree, at bars that the expansions' own error does not hide: the
U list's windows of 64 leaves and chunks of 512 points, and the frequency-domain translations on trees of
one tile to many, with the transposed evaluation tied to them by <g, A q> = <A^T g, q>.

Both evaluators compute the same sums on the same operators up to the order of their terms; the check-to-
equivalent maps amplify that rounding by up to 1e3 for m <= 6 and 1e7 at m = 10 and 14, so that 1e-10 of
the near field's sums (m = 4) and 1e-9 and 1e-7 of the translations' allow it with a factor of ten and
more.  A source left out, a wrong partner or a lost product is 1e-6 and above."""
import numpy as np
import pytest

import oracle as O
import pvfmm_amd as P

from test_hadamard_runs import points

pytestmark = pytest.mark.gpu


def _oracle(src, trg, max_pts, kernel, m, dens):
    t = O.OracleTree(src, trg, max_pts)
    t.set_operators(O.precompute(kernel, m))
    return [np.asarray(t.evaluate(q)).ravel() for q in dens]


@pytest.mark.parametrize("kernel,n,max_pts,n_trg", [
    ("laplace_poten", 600, 2, 0),      # one point to a leaf: windows of 64 points
    ("laplace_grad", 900, 3, 0),
    ("stokes_vel", 500, 2, 0),
    ("laplace_poten", 512, 512, 0),    # a chunk's points
    ("laplace_grad", 513, 600, 0),
    ("laplace_grad", 3000, 700, 0),    # leaves of more than a block's targets
    ("stokes_vel", 1500, 400, 0),
    ("laplace_poten", 700, 4, 2500),   # leaves without sources within a window
    ("laplace_grad", 40, 8, 4000),
])
def test_u_list_windows(gpu, kernel, n, max_pts, n_trg):
    rng = np.random.default_rng(n + max_pts)
    x = np.concatenate([rng.random((n - n // 4, 3)), 0.7 + 0.01 * rng.random((n // 4, 3))])
    y = rng.random((n_trg, 3)) if n_trg else x
    q = rng.standard_normal(P.kernel_dims(kernel)[0] * n)
    u = P.PtFMMTree(x, y, max_pts).setup(P.PtFMM(kernel, 4, "fp64")).evaluate(q)
    ref, = _oracle(x, y, max_pts, kernel, 4, [q])
    e = float(np.linalg.norm(u - ref) / np.linalg.norm(ref))
    assert e < 1e-10, e


@pytest.mark.parametrize("m,kind,n,max_pts,nv", [
    (4, "uniform", 6000, 60, 1),   # 196 products: a block per tile
    (6, "uniform", 1500, 60, 1),   # one tile of 8 targets
    (6, "uniform", 6000, 60, 1),   # two tiles
    (6, "shell", 60000, 40, 1),    # runs of tiles
    (4, "shell", 90000, 30, 3),
    (6, "cluster", 40000, 25, 2),
    (10, "cluster", 20000, 100, 1),
    (14, "cluster", 3000, 60, 1),  # the transforms of any m
])
def test_fp64_translations(gpu, m, kind, n, max_pts, nv):
    import torch

    x = points(kind, n)
    rng = np.random.default_rng(6)
    q, g = rng.standard_normal((nv, n)), rng.standard_normal((nv, n))
    t = P.PtFMMTree(x, x, max_pts).setup(P.PtFMM("laplace_poten", m, "fp64"), n_vec_max=nv)
    u, a = (f(torch.tensor(v if nv > 1 else v[0], device="cuda:0")).reshape(nv, n).cpu().numpy()
            for f, v in ((t.evaluate_device, q), (t.evaluate_adjoint_device, g)))
    tol = 1e-9 if m <= 6 else 1e-7
    for v, ref in enumerate(_oracle(x, x, max_pts, "laplace_poten", m, q)):
        e = float(np.linalg.norm(u[v] - ref) / np.linalg.norm(ref))
        d = float(abs(g[v] @ u[v] - a[v] @ q[v]) / (np.linalg.norm(g[v]) * np.linalg.norm(u[v])))
        print(f"m = {m}, {kind} {n}, vector {v}: {e:.2e} from the oracle, adjoint {d:.2e}")
        assert e < tol and d < tol, (v, e, d)
