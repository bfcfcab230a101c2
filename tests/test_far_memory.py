"""Far rows split over blocks keep one sum per segment and target: in a tree of large leaves, where
nearly every row with W items is long, these sums may not outgrow the outputs without bound."""
import numpy as np
import pytest

import oracle as O
import pvfmm_amd as P
from pvfmm_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_segment_sums_stay_within_four_times_the_outputs(gpu):
    rng = np.random.default_rng(5)
    n, m, nv = 500000, 4, 8
    x = np.concatenate([0.3 + 0.01 * rng.standard_normal((n - n // 10, 3)), W.uniform(rng, n // 10)])
    t = P.PtFMMTree(x, x, 10000)
    fmm = P.PtFMM("laplace_grad", m, "mixed")
    one = t.setup(fmm, n_vec_max=1).stats()["device_bytes"]
    s = t.setup(fmm, n_vec_max=nv).stats()
    K, nodes = 6 * (m - 1) ** 2 + 2, s["n_nodes"]
    # per vector: densities and outputs, equivalent and check densities of the boxes and leaves, spectra
    rows = 3 * nodes + 2 * max(s["s2m_rows"], s["l2t_rows"])
    own = 4 * n + 24 * n + 4 * K * (rows + s["l2t_rows"]) + 64 * m * (2 * m - 1) ** 2 * (s["v_src_slots"] + s["v_trg_slots"])
    work = 4 * 2**25  # partial products of the translations, for all vectors
    sums = (s["device_bytes"] - one - work) / (nv - 1) - 1.02 * own
    print(f"per vector: outputs {24 * n / 2**20:.1f} MiB, beyond the other buffers at least {sums / 2**20:.1f} MiB")
    assert sums < 4 * 24 * n  # 16 times the outputs when not bounded
    q = rng.standard_normal((nv, n))
    u = t.evaluate(q)
    idx = rng.choice(n, 300, replace=False)
    for v in (0, nv - 1):
        ref = O.direct("laplace_grad", x, q[v], x[idx]).ravel()
        got = u[v].reshape(n, 3)[idx].ravel()
        e = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
        assert e < 1e-2, (v, e)  # m = 4: 1e-3
