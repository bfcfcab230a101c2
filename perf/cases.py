"""The calls that a user of this framework times: FMM evaluations through its public entry points.

A case names the entry point ("call"), the kernel, the points' distribution and number, the
multipole order m, max_pts, the precision and what else the entry point takes:

* "tree": ``PtFMMTree.setup(PtFMM(...))`` once, then ``evaluate_device`` of new density vectors
  on the GPU: one step of a solver on a fixed geometry (its matrix-vector product).
* "batch": many independent clouds through one ``PtFMMBatch.evaluate_device``.
* "grad": ``LaplaceFMM`` behind torch.autograd, the forward evaluation and the gradients with
  respect to positions and charges.
* "context": ``FMMParticleContext.evaluate`` on host arrays, the interface of the reference's
  own bindings: with setup=True (its default) for points that moved, with setup=False for new
  densities on the same points.

The mixed evaluator computes in FP32, so a program that chooses it keeps its results in FP32:
those cases return float32 values.  Launch shapes are the defaults (no autotune call).
"""
import math

import numpy as np
import torch

import pvfmm_amd as P
from pvfmm_amd import workloads as W
from pvfmm_amd.autograd import LaplaceFMM

_DIMS = {"laplace_poten": (1, 1), "laplace_grad": (1, 3), "stokes_vel": (3, 3)}
_ENUM = {"laplace_poten": P.FMMKernel.LaplacePotential, "laplace_grad": P.FMMKernel.LaplaceGradient,
         "stokes_vel": P.FMMKernel.StokesVelocity}
_PAIR_FLOPS = {"laplace_poten": 9, "laplace_grad": 16, "stokes_vel": 29}


def listed():
    return [
        # the smallest call: a few thousand points, where launches and latency are all the time
        dict(name="poten-fp64-4k", call="tree", kernel="laplace_poten", points="uniform", n=4099, m=6, max_pts=100,
             precision="fp64"),
        # an ordinary FP64 call: the reference's first example (uniform points, m = 6)
        dict(name="poten-fp64-64k", call="tree", kernel="laplace_poten", points="uniform", n=65536, m=6, max_pts=128,
             precision="fp64"),
        # the headline workload: a strongly adaptive tree, the gradient kernel, high order, FP32
        dict(name="grad-mixed-2m", call="tree", kernel="laplace_grad", points="adaptive", n=2097152, m=10, max_pts=256,
             precision="mixed"),
        # its FP64 counterpart, for users who need ten digits
        dict(name="grad-fp64-1m", call="tree", kernel="laplace_grad", points="adaptive", n=1000003, m=10, max_pts=256,
             precision="fp64"),
        # boundary-integral Stokes flow: forces on a closed surface, FP32
        dict(name="stokes-mixed-1m", call="tree", kernel="stokes_vel", points="ellipsoid", n=1048576, m=8, max_pts=200,
             precision="mixed"),
        # velocities off the surface (targets other than the sources) in FP64, a ragged size
        dict(name="stokes-fp64-150k", call="tree", kernel="stokes_vel", points="ellipsoid", n=150001, n_trg=70003, m=6,
             max_pts=150, precision="fp64"),
        # block Krylov or many right-hand sides: 32 density vectors on one tree
        dict(name="densities-32-1m", call="tree", kernel="laplace_poten", points="uniform", n=1048576, m=8, max_pts=128,
             precision="mixed", n_vec=32),
        # the periodic box of a particle simulation
        dict(name="periodic-mixed-1m", call="tree", kernel="laplace_poten", points="uniform", n=1048576, m=8, max_pts=128,
             precision="mixed", bndry="pxyz"),
        # many independent small problems in one launch
        dict(name="clouds-24", call="batch", kernel="laplace_poten", n_clouds=24, log2_min=11.0, log2_max=16.0, m=8,
             max_pts=128, precision="mixed"),
        # training or force matching: energy forward, gradients for positions and charges
        dict(name="energy-grad-260k", call="grad", of="energy", points="uniform", n=262147, m=10, max_pts=256,
             precision="mixed"),
        # a time step with moved points on host arrays: tree, lists, plan and evaluation
        dict(name="context-moved-100k", call="context", kernel="stokes_vel", points="uniform", n=100003, m=6, max_pts=150,
             dtype="float32", setup=True),
        # further densities on the same points from host arrays, FP64
        dict(name="context-same-300k", call="context", kernel="laplace_grad", points="adaptive", n=300007, m=8, max_pts=200,
             dtype="float64", setup=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["tree", "tree", "tree", "tree", "batch", "grad", "context", "context"])
    kernel = rng.choice(["laplace_poten", "laplace_grad", "stokes_vel"])
    points = rng.choice(["uniform", "adaptive", "ellipsoid"])
    if call == "batch":
        return dict(call=call, kernel="laplace_poten", n_clouds=rng.randint(2, 24), log2_min=11.0,
                    log2_max=round(rng.uniform(12.0, 16.0), 3), m=rng.choice([6, 8, 10]), max_pts=rng.randint(64, 200),
                    precision=rng.choice(["mixed", "fp64"]))
    if call == "grad":
        return dict(call=call, of=rng.choice(["energy", "potential"]), points=rng.choice(["uniform", "adaptive"]),
                    n=_log_int(rng, 4000, 300000), m=rng.choice([6, 8, 10]), max_pts=rng.randint(100, 300),
                    precision=rng.choice(["mixed", "fp64"]))
    if call == "context":
        setup = rng.choice([True, False])
        return dict(call=call, kernel=kernel, points=points, n=_log_int(rng, 4000, 200000 if setup else 400000),
                    m=rng.choice([4, 6] if kernel == "stokes_vel" else [4, 6, 8]), max_pts=rng.randint(80, 250),
                    dtype=rng.choice(["float32", "float64"]), setup=setup)
    case = dict(call=call, kernel=kernel, points=points, n=0, m=0, max_pts=rng.randint(80, 300),
                precision=rng.choice(["mixed", "mixed", "fp64"]))
    if kernel == "stokes_vel":
        # FP64 Stokes up to m = 6: from m = 8 on its check-to-equivalent cutoff keeps directions that
        # amplify rounding to 1e-5 of the result, and such users take the mixed evaluator
        mixed = case["precision"] == "mixed"
        case.update(m=rng.choice([4, 6, 8] if mixed else [4, 6]), n=_log_int(rng, 4000, 800000 if mixed else 200000))
    else:
        case.update(m=rng.choice([4, 6, 8, 10]), n=_log_int(rng, 4000, 1500000 if case["precision"] == "mixed" else 700000))
    more = rng.choice(["", "", "targets", "vectors", "periodic"])
    if more == "targets":
        case["n_trg"] = _log_int(rng, max(1000, case["n"] // 8), case["n"])
    elif more == "vectors" and kernel == "laplace_poten":
        case["n_vec"] = rng.choice([2, 3, 5, 8, 13, 16])
        case["n"] = min(case["n"], 2000000 // case["n_vec"])
    elif more == "periodic" and kernel == "laplace_poten" and case["m"] < 10:
        case["bndry"] = "pxyz"
    return case


# ----------------------------------------------------------------------------- inputs
def _points(rng, kind, n):
    if kind == "uniform":
        return W.uniform(rng, n)
    if kind == "ellipsoid":
        return W.ellipsoid_surface(rng, n)
    n_s, n_g = n // 2, int(0.3 * n)
    return np.concatenate([W.sphere_surface(rng, n_s), W.gaussian_blob(rng, n_g), W.uniform(rng, n - n_s - n_g)])


def _inputs(case, seed):
    """The case's host inputs: (src, trg or None, densities) or, for a batch, a list of (src, den)."""
    rng = np.random.default_rng([7, seed])
    if case["call"] == "batch":
        sizes = np.floor(2.0 ** np.linspace(case["log2_min"], case["log2_max"], case["n_clouds"])).astype(int)
        return [(W.uniform(rng, int(s)), rng.standard_normal(int(s))) for s in sizes]
    k0 = _DIMS[case.get("kernel", "laplace_poten")][0]
    src = _points(rng, case["points"], case["n"])
    # targets other than the sources: points of the box around them
    trg = W.uniform(rng, case["n_trg"]) if case.get("n_trg") else None
    nv = case.get("n_vec", 1)
    return src, trg, rng.standard_normal((nv, k0 * case["n"]) if nv > 1 else k0 * case["n"])


def prepare(case, seed):
    if case["call"] == "batch":
        clouds = _inputs(case, seed)
        fmm = P.PtFMM(case["kernel"], case["m"], case["precision"])
        trees = [P.PtFMMTree(x, x, case["max_pts"]).setup(fmm) for x, _ in clouds]
        return dict(case=case, fmm=fmm, batch=P.PtFMMBatch(trees), den=[torch.from_numpy(q).to("cuda") for _, q in clouds])
    src, trg, den = _inputs(case, seed)
    if case["call"] == "tree":
        fmm = P.PtFMM(case["kernel"], case["m"], case["precision"])
        tree = P.PtFMMTree(src, trg, case["max_pts"], bndry=case.get("bndry", "free"))
        tree.setup(fmm, n_vec_max=case.get("n_vec", 1))
        return dict(case=case, fmm=fmm, tree=tree, den=torch.from_numpy(den).to("cuda"))
    if case["call"] == "grad":
        fmm = LaplaceFMM(src, case["m"], case["max_pts"], case["precision"])
        g = np.random.default_rng([8, seed]).standard_normal(case["n"])
        return dict(case=case, fmm=fmm, x=torch.from_numpy(src).to("cuda").requires_grad_(),
                    q=torch.from_numpy(den).to("cuda").requires_grad_(), g=torch.from_numpy(g).to("cuda"))
    dt = np.dtype(case["dtype"])
    ctx = P.FMMParticleContext(-1.0, case["max_pts"], case["m"], _ENUM[case["kernel"]], dtype=dt)
    x, den = src.astype(dt).ravel(), _context_densities(case, den).astype(dt)
    if not case["setup"]:
        ctx.evaluate(x, den, None, x, setup=True)
    return dict(case=case, ctx=ctx, x=x, den=den)


def _context_densities(case, den):
    # the context's density arrays are as long as the source positions, whatever the kernel takes
    return np.concatenate([den, np.zeros(3 * case["n"] - len(den))])


def run(state):
    case = state["case"]
    if case["call"] == "tree":
        return _kept(case, state["tree"].evaluate_device(state["den"]))
    if case["call"] == "batch":
        return [_kept(case, o) for o in state["batch"].evaluate_device(state["den"])]
    if case["call"] == "context":
        return state["ctx"].evaluate(state["x"], state["den"], None, state["x"], setup=case["setup"])
    fmm, x, q = state["fmm"], state["x"], state["q"]
    if case["of"] == "energy":
        e = fmm.energy(x, q)
        gx, gq = torch.autograd.grad(e, (x, q))
    else:
        e = fmm.potential(x, q)
        gx, gq = torch.autograd.grad(e, (x, q), state["g"])
    return [_kept(case, t) for t in (e.detach(), gx, gq)]


def _kept(case, t):
    return t.float() if case["precision"] == "mixed" else t


# ----------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Bytes of the densities, coordinates and results, and the flops of an FMM on a uniform tree
    with leaves half full: the near field over 27 leaves, the surfaces of the leaves twice, the
    26 parent offsets of the frequency products and the translations up and down."""
    if case["call"] == "batch":
        sizes = np.floor(2.0 ** np.linspace(case["log2_min"], case["log2_max"], case["n_clouds"]))
        parts = [_work(case["kernel"], s, s, case["m"], case["max_pts"], 1) for s in sizes]
        return {k: float(sum(p[k] for p in parts)) for k in ("bytes", "flops")}
    n, kernel = case["n"], case.get("kernel", "laplace_poten")
    w = _work(kernel, n, case.get("n_trg", n), case["m"], case["max_pts"], case.get("n_vec", 1))
    if case["call"] == "grad":
        b = _work("laplace_grad", n, n, case["m"], case["max_pts"], 1 if case["of"] == "energy" else 2)
        w = {k: 2 * w[k] + b[k] for k in w}
    return {k: float(v) for k, v in w.items()}


def _work(kernel, n, n_trg, m, max_pts, nv):
    k0, k1 = _DIMS[kernel]
    e1 = 3 if kernel == "stokes_vel" else 1
    per_leaf = max_pts / 2
    leaves, ns = n / per_leaf, 6 * (m - 1) ** 2 + 2
    pairs = 27 * per_leaf * n_trg + ns * (n + n_trg)
    spectra = leaves / 8 * 26 * 4 * m * m * (m + 1) * 512 * k0 * e1
    gemms = 6 * leaves * 2 * (ns * k0) ** 2
    coords = 24 * (n + n_trg)
    return {"bytes": nv * 8 * (k0 * n + k1 * n_trg) + coords, "flops": nv * (_PAIR_FLOPS[kernel] * pairs + spectra + gemms)}


# ----------------------------------------------------------------------------- 64-bit results
_MOST_PAIRS = 1.2e11  # direct sums of more pairs take too long


def _direct(kernel, src, den, trg):
    """The kernel's sum over all sources for all targets in 64 bits, coincident pairs left out."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    s, t = (torch.as_tensor(a, dtype=torch.float64, device=dev).reshape(-1, 3) for a in (src, trg))
    k0, k1 = _DIMS[kernel]
    f = torch.as_tensor(den, dtype=torch.float64, device=dev).reshape(-1, k0)
    out = torch.empty((len(t), k1), dtype=torch.float64, device=dev)
    step = max(1, int(1.5e8 // max(1, len(s))))
    for i in range(0, len(t), step):
        d = [t[i:i + step, a, None] - s[None, :, a] for a in range(3)]
        r2 = d[0] * d[0]
        r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        r = torch.where(r2 > 0, r2, torch.inf).rsqrt_()
        if kernel == "laplace_poten":
            out[i:i + step, 0] = r @ f[:, 0]
        elif kernel == "laplace_grad":
            r.pow_(3)
            for a in range(3):
                out[i:i + step, a] = d[a].mul_(r) @ f[:, 0]
        else:
            ip = d[0] * f[:, 0]
            ip.addcmul_(d[1], f[None, :, 1]).addcmul_(d[2], f[None, :, 2])
            free = r @ f
            ip.mul_(r).mul_(r).mul_(r)
            for a in range(3):
                out[i:i + step, a] = free[:, a] + d[a].mul_(ip).sum(1)
    return out * (1 / (8 * math.pi) if kernel == "stokes_vel" else 1 / (4 * math.pi))


def exact(case, seed):
    if case["call"] == "batch":
        clouds = _inputs(case, seed)
        if sum(len(q) ** 2 for _, q in clouds) > _MOST_PAIRS:
            return None
        return [_direct(case["kernel"], x, q, x).reshape(-1) for x, q in clouds]
    n, nv = case["n"], case.get("n_vec", 1)
    if float(n) * case.get("n_trg", n) * nv > _MOST_PAIRS or case.get("bndry", "free") != "free":
        return None
    src, trg, den = _inputs(case, seed)
    if case["call"] == "context":
        # the sum over the positions and densities that the context was given
        src = src.astype(case["dtype"]).astype(np.float64)
        u = _direct(case["kernel"], src, den.astype(case["dtype"]), src).reshape(-1)
        return torch.cat([u, u.new_zeros(3 * n - len(u))])
    if case["call"] == "tree":
        trg = src if trg is None else trg
        u = [_direct(case["kernel"], src, d, trg).reshape(-1) for d in np.atleast_2d(den)]
        return torch.stack(u) if nv > 1 else u[0]
    q = den
    phi, field = _direct("laplace_poten", src, q, src)[:, 0], _direct("laplace_grad", src, q, src)
    tq = torch.as_tensor(q, device=phi.device)
    if case["of"] == "energy":
        return [0.5 * torch.dot(tq, phi), -tq[:, None] * field, phi]
    g = np.random.default_rng([8, seed]).standard_normal(n)
    tg = torch.as_tensor(g, device=phi.device)
    back = _direct("laplace_grad", src, g, src)
    return [phi, -(tg[:, None] * field + tq[:, None] * back), _direct("laplace_poten", src, g, src)[:, 0]]
