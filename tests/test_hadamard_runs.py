"""GPU: the FP64 frequency-domain translations of the scalar kernels, whose blocks take equal shares of
the (pair of frequencies, tile) products, on trees with one tile, a few and many, full and ragged, with
groups that lack partners, and with several vectors; fewer than 512 products take a block per tile.
The reference is the FP32 path (other kernels and another layout of the tiles), whose rounding allows
1e-5 of the largest value at every target; FP64 against the direct sum at the accuracy of m where the
number of points is small."""
import numpy as np
import pytest

import pvfmm_amd as P

pytestmark = pytest.mark.gpu


def points(kind, n, seed=5):
    rng = np.random.default_rng(seed)
    if kind == "uniform":
        return rng.random((n, 3))
    if kind == "shell":  # nonuniform: groups of targets without a partner at many offsets
        v = rng.standard_normal((n, 3))
        return 0.5 + v / np.linalg.norm(v, axis=1)[:, None] * np.array([0.45, 0.2, 0.1])
    return np.concatenate([rng.random((n // 2, 3)), 0.3 + 0.02 * rng.random((n - n // 2, 3))])


@pytest.mark.parametrize("m,kind,n,max_pts,nv,bndry", [
    (4, "uniform", 6000, 60, 1, "free"),   # 196 products: a block per tile
    (6, "uniform", 1500, 60, 1, "free"),   # one tile of 8 targets
    (6, "uniform", 6000, 60, 1, "free"),   # two tiles
    (10, "cluster", 20000, 100, 1, "free"),
    (6, "shell", 60000, 40, 1, "free"),
    (4, "shell", 90000, 30, 3, "free"),
    (6, "uniform", 20000, 60, 2, "pxyz"),
    (14, "cluster", 3000, 60, 1, "free"),  # the transforms of any m
])
def test_fp64_translations(m, kind, n, max_pts, nv, bndry):
    import torch

    x = points(kind, n)
    rng = np.random.default_rng(6)
    q = torch.tensor(rng.standard_normal((nv, n)), device="cuda:0")
    if bndry != "free":
        q -= q.mean(dim=1, keepdim=True)
    u = {}
    for prec in ("fp64", "mixed"):
        f = P.PtFMM("laplace_poten", m, prec)
        t = P.PtFMMTree(x, x, max_pts, bndry=bndry).setup(f, n_vec_max=nv)
        u[prec] = t.evaluate_device(q if nv > 1 else q[0].contiguous()).reshape(nv, n)
        a = t.evaluate_adjoint_device(q if nv > 1 else q[0].contiguous()).reshape(nv, n)
        u[prec + " adjoint"] = a
    for k in ("", " adjoint"):
        for v in range(nv):
            e = float((u["fp64" + k][v] - u["mixed" + k][v]).abs().max() / u["fp64" + k][v].abs().max())
            assert e < 1e-5, (k, v, e)
    if n <= 6000:
        ref = P.direct("laplace_poten", x, q[0].cpu().numpy(), x)
        e = np.linalg.norm(u["fp64"][0].cpu().numpy() - ref) / np.linalg.norm(ref)
        assert e < {4: 1e-2, 6: 1e-4, 14: 1e-8}[m], e
