"""Trees set up with one PtFMM share its operators on the device.  Their results must be those
of a tree with a handle of its own, bit for bit, whatever was set up before on the shared handle
(another point set, a periodic tree, the adjoint, many vectors), from several threads, and a
context that changes precision must not keep the operators of the old one."""
import threading

import numpy as np
import pytest

import pvfmm_amd as P

pytestmark = pytest.mark.gpu


def _run(fmm, kernel, seed, bndry="free", n=1500):
    rng = np.random.default_rng(seed)
    k0, k1 = P.kernel_dims(kernel)
    x = rng.random((n + 37 * seed, 3))
    t = P.PtFMMTree(x, x, 40, bndry=bndry).setup(fmm)
    u = t.evaluate(rng.standard_normal(k0 * len(x)))
    a = t.evaluate_adjoint(rng.standard_normal(k1 * len(x))) if kernel != "laplace_grad" else np.zeros(0)
    return np.concatenate([u, a])


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kernel,m", [("laplace_poten", 4), ("laplace_grad", 6), ("stokes_vel", 4)])
def test_shared_handle_gives_the_results_of_its_own(gpu, kernel, m, prec):
    shared = P.PtFMM(kernel, m, prec)
    cases = [(1, "free"), (2, "pxyz"), (3, "free"), (4, "px"), (1, "free")]
    own = [_run(P.PtFMM(kernel, m, prec), kernel, s, b) for s, b in cases]
    for (s, b), ref in zip(cases, own):
        assert np.array_equal(_run(shared, kernel, s, b), ref), (s, b)


def test_first_setup_from_several_threads(gpu):
    shared = P.PtFMM("laplace_poten", 6, "mixed")
    got = [None] * 6

    def work(i):
        got[i] = _run(shared, "laplace_poten", i % 3)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(6):
        assert np.array_equal(got[i], _run(P.PtFMM("laplace_poten", 6, "mixed"), "laplace_poten", i % 3)), i


def test_context_that_changes_precision(gpu):
    from pvfmm_amd import ffi

    rng = np.random.default_rng(5)
    x, q = rng.random(3 * 900), rng.standard_normal(3 * 900)
    ctx = P.FMMParticleContext(-1.0, 40, 6, P.FMMKernel.StokesVelocity)
    a = ctx.evaluate(x, q, None, x)
    ffi.check(ffi.lib().PVFMMSetMixedPrecision(ctx._ptr, 1))
    b = ctx.evaluate(x, q, None, x)
    ffi.check(ffi.lib().PVFMMSetMixedPrecision(ctx._ptr, 0))
    assert np.array_equal(ctx.evaluate(x, q, None, x), a)
    fresh = P.FMMParticleContext(-1.0, 40, 6, P.FMMKernel.StokesVelocity, mixed_precision=True)
    assert np.array_equal(fresh.evaluate(x, q, None, x), b)
    assert not np.array_equal(a, b)
