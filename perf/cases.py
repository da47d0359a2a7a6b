"""Workloads of the 2-D FMM package for timing: what a user's program asks of
it, through the public classes and functions.

A case is a dict of plain values:

* ``method``   laplace, dipole, helmholtz, stokes, stokes_dipole, blackbox
* ``mode``     what one pass is
    - ``solve``  points, densities and targets are new: tree, expansions and
      evaluation (a time step of moving points, a one-off sum);
    - ``apply``  the tree stays, the densities are new: expansions and
      self-evaluation (one product of an iterative solver);
    - ``probe``  the expansions stay, the targets are new: potential and
      gradient at them (field lines, plots, particle tracing);
    - ``train``  forward and backward of a squared misfit through the
      differentiable functions.
* ``points``   uniform (the unit square), clusters (Gaussian), circle (a curve)
* ``n``, ``targets`` (self, grid, uniform), ``nt``
* ``p``        equivalent points per box (Chebyshev order for blackbox)
* ``ncut``     leaf capacity
* ``precision``

The root box is the unit square throughout, so that every pass meets the same
box widths whatever ran before it.
"""
import math

import torch

from flexmm_amd import kernels
from flexmm_amd.flexmm2d import BB_FMM
from flexmm_amd.kifmm2d import FMM, StokesFMM, fmm_evaluate, stokes_evaluate

BOX = [0.0, 1.0, 0.0, 1.0]
WAVENUMBER = 20.0
FOUR_PI, TWO_PI = 4.0 * math.pi, 2.0 * math.pi


def _case(method, mode, points, n, targets, nt, p, ncut, precision="fp64"):
    return dict(method=method, mode=mode, points=points, n=n, targets=targets, nt=nt, p=p,
                ncut=ncut, precision=precision)


def listed():
    def c(name, *a, **k):
        return dict(_case(*a, **k), name=name)

    return [
        # a small self-evaluation from scratch: the latency of the whole chain
        c("laplace_small", "laplace", "solve", "uniform", 2003, "self", 2003, 32, 64),
        # the CPU-sized problem of the tests
        c("laplace_100k_self", "laplace", "solve", "uniform", 100_000, "self", 100_000, 32, 64),
        # the headline: 1M sources to a 1000 x 1000 grid, FP64 and mixed
        c("laplace_1m_grid", "laplace", "solve", "uniform", 1_000_000, "grid", 1_000_000, 60, 100),
        c("laplace_1m_grid_mixed", "laplace", "solve", "uniform", 1_000_000, "grid", 1_000_000,
          60, 100, precision="mixed"),
        # a deep adaptive tree under a grid of targets
        c("laplace_1m_clusters", "laplace", "solve", "clusters", 1_000_000, "grid", 1_000_000,
          60, 100),
        # an iterative solver's matrix-vector product at the sizes of the
        # reference's Laplace example (N 50,000, Nequiv 64, Ncutoff 500)
        c("laplace_apply_50k", "laplace", "apply", "uniform", 50_000, "self", 50_000, 64, 500),
        # a boundary-integral product: single + double layer on a curve, odd size
        c("dipole_apply_curve", "dipole", "apply", "circle", 100_003, "self", 100_003, 60, 100),
        # potential and gradient at new points off a curve of sources
        c("laplace_probe", "laplace", "probe", "circle", 300_007, "uniform", 20_011, 60, 100),
        # differentiable modified Helmholtz: forward, d/dcharges, d/dpositions
        c("helmholtz_train", "helmholtz", "train", "circle", 500_000, "uniform", 200_000, 60, 100),
        # black-box FMM at its defaults (order 8, Ncutoff 50) on the headline points
        c("blackbox_1m_grid", "blackbox", "solve", "uniform", 1_000_000, "grid", 1_000_000, 8, 50),
        # Stokeslets: 2M forces in clusters, self-evaluation, forward and adjoint
        c("stokes_2m_train", "stokes", "train", "clusters", 2_000_000, "self", 2_000_000, 64, 100,
          precision="mixed"),
        # Stokeslets + stresslets, FP64, velocity and pressure
        c("stokes_dipole_300k", "stokes_dipole", "solve", "clusters", 300_001, "self", 300_001,
          64, 100),
    ]


_MODES = {"laplace": ("solve", "solve", "apply", "probe", "train"),
          "dipole": ("solve", "apply"),
          "helmholtz": ("solve", "apply", "probe", "train"),
          "stokes": ("solve", "apply", "train"),
          "stokes_dipole": ("solve", "apply"),
          "blackbox": ("solve", "apply")}


def draw(rng):
    """A case of the ranges that the listed ones stand for."""
    most = max(work(c)["flops"] for c in listed())

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        method = rng.choice(["laplace", "laplace", "laplace", "dipole", "helmholtz", "stokes",
                             "stokes_dipole", "blackbox"])
        mode = rng.choice(_MODES[method])
        points = rng.choice(["uniform", "clusters", "circle"])
        n = size(1000, 1_000_000)
        if method in ("dipole", "stokes", "stokes_dipole") or mode == "apply":
            targets = "self"
        elif mode in ("probe", "train"):
            targets = "uniform"
        else:
            targets = rng.choice(["self", "grid", "uniform"])
        nt = n
        if targets == "uniform":
            nt = size(1000, 1_000_000)
        elif targets == "grid":
            nt = size(32, 1000) ** 2
        p = rng.randint(4, 8) if method == "blackbox" else rng.choice([32, 48, 60, 64])
        ncut = rng.choice([50, 64, 100, 100, 200] + ([500] if n >= 20_000 else []))
        precision = "fp64"
        if method in ("laplace", "stokes") and mode != "probe":
            precision = rng.choice(["fp64", "fp64", "mixed"])
        case = _case(method, mode, points, n, targets, nt, p, ncut, precision)
        if work(case)["flops"] <= 0.5 * most:
            return case


# -- inputs --------------------------------------------------------------------

def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, n):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _randn(g, n):
    return torch.randn(n, generator=g, device="cuda", dtype=torch.float64)


def _points(g, kind, n):
    if kind == "uniform":
        return _rand(g, n), _rand(g, n)
    if kind == "circle":
        th = TWO_PI * _rand(g, n)
        return 0.5 + 0.4 * torch.cos(th), 0.5 + 0.4 * torch.sin(th)
    nc = max(3, min(100, n // 20_000))
    cx, cy = 0.1 + 0.8 * _rand(g, nc), 0.1 + 0.8 * _rand(g, nc)
    which = (_rand(g, n) * nc).long().clamp_(max=nc - 1)
    x = cx[which] + 0.005 * _randn(g, n)
    y = cy[which] + 0.005 * _randn(g, n)
    return x.clamp_(0.0, 1.0), y.clamp_(0.0, 1.0)


def _inputs(case, seed):
    g = _rng(seed)
    n, nt, method = case["n"], case["nt"], case["method"]
    s = {"case": case}
    s["x"], s["y"] = _points(g, case["points"], n)
    if case["targets"] == "self":
        s["tx"], s["ty"] = s["x"], s["y"]
    elif case["targets"] == "grid":
        m = math.isqrt(nt)
        a = torch.linspace(0.0, 1.0, m, device="cuda", dtype=torch.float64)
        gx, gy = torch.meshgrid(a, a, indexing="ij")
        s["tx"], s["ty"] = gx.reshape(-1).contiguous(), gy.reshape(-1).contiguous()
    else:
        s["tx"], s["ty"] = _rand(g, nt), _rand(g, nt)
    if method in ("stokes", "stokes_dipole"):
        s["f"] = [_randn(g, n) for _ in range(2)]
        if method == "stokes_dipole":
            th = TWO_PI * _rand(g, n)
            s["f"] += [_randn(g, n), _randn(g, n), torch.cos(th), torch.sin(th)]
        if case["mode"] == "train":
            s["goal"] = [math.sqrt(n) * _randn(g, nt) for _ in range(2)]
    elif method == "dipole":
        th = TWO_PI * _rand(g, n)
        s["tau"] = torch.stack([_randn(g, n), _randn(g, n)])
        s["normal"] = torch.stack([torch.cos(th), torch.sin(th)])
    else:
        s["tau"] = _randn(g, n)
        if case["mode"] == "train":
            s["goal"] = math.sqrt(n) * _randn(g, nt)
    return s


def _kernel(case):
    if case["method"] == "helmholtz":
        return kernels.modified_helmholtz(WAVENUMBER)
    return kernels.laplace, kernels.laplace_potential, kernels.laplace_gradient


def _fmm(s):
    case = s["case"]
    if case["method"] == "blackbox":
        return BB_FMM(s["x"], s["y"], kernels.laplace, Ncutoff=case["ncut"], p=case["p"], bbox=BOX,
                      precision=case["precision"])
    if case["method"] in ("stokes", "stokes_dipole"):
        return StokesFMM(s["x"], s["y"], case["p"], case["ncut"], bbox=BOX,
                         precision=case["precision"])
    f = FMM(s["x"], s["y"], _kernel(case)[0], case["ncut"], case["p"], bbox=BOX,
            precision=case["precision"])
    if case["method"] == "dipole":
        f.register_upwardor(kernels.laplace_slp_dlp, "slp+dlp")
        f.register_evaluator(f.helper.functions["kernel_app"], kernels.laplace_slp_dlp,
                             "slp+dlp->u", 1)
    return f


def _expand(f, s):
    method = s["case"]["method"]
    if method == "stokes":
        f.build_expansions(*s["f"])
    elif method == "stokes_dipole":
        f.build_expansions_dipole(*s["f"])
    elif method == "dipole":
        f.build_expansions(s["tau"], "slp+dlp", s["normal"])
    else:
        f.build_expansions(s["tau"])


def _evaluate(f, s):
    method, own = s["case"]["method"], s["case"]["targets"] == "self"
    tx, ty = s["tx"], s["ty"]
    if method == "stokes":
        return f.evaluate_to_points(tx, ty, own)
    if method == "stokes_dipole":
        return f.evaluate_to_points_dipole(tx, ty, own)
    if method == "dipole":
        return f.evaluate_to_points(tx, ty, "slp+dlp->u", own)
    return f.source_evaluation(tx, ty) if own else f.target_evaluation(tx, ty)


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["mode"] in ("apply", "probe"):
        s["fmm"] = _fmm(s)      # the tree that such a program keeps
    if case["mode"] == "probe":
        _, _, grad = _kernel(case)
        s["fmm"].register_evaluator(grad, grad, "gradient", 3)
        _expand(s["fmm"], s)
    return s


def run(s):
    case = s["case"]
    mode = case["mode"]
    if mode == "apply":
        _expand(s["fmm"], s)
        return _evaluate(s["fmm"], s)
    if mode == "probe":
        return s["fmm"].evaluate_to_points(s["tx"], s["ty"], "gradient", False)
    if mode == "solve":
        f = _fmm(s)
        _expand(f, s)
        u = _evaluate(f, s)
        f.close()
        return u
    own = case["targets"] == "self"
    if case["method"] == "stokes":
        fx, fy = (a.detach().requires_grad_(True) for a in s["f"])
        u, v = stokes_evaluate(s["x"], s["y"], fx, fy, s["tx"], s["ty"], case["p"], case["ncut"],
                               bbox=BOX, precision=case["precision"], check=own)
        loss = ((u - s["goal"][0]) ** 2).sum() + ((v - s["goal"][1]) ** 2).sum()
        return (u.detach(), v.detach()) + torch.autograd.grad(loss, (fx, fy))
    x, y, tau = (s[k].detach().requires_grad_(True) for k in ("x", "y", "tau"))
    u = fmm_evaluate(x, y, tau, s["tx"], s["ty"], _kernel(case)[0], case["ncut"], case["p"],
                     bbox=BOX, precision=case["precision"], check=own)
    loss = ((u - s["goal"]) ** 2).sum()
    return (u.detach(),) + torch.autograd.grad(loss, (x, y, tau))


# -- the work of a pass ----------------------------------------------------------

# floating-point operations of one source-target pair (potential, with gradient)
_PAIR = {"laplace": (20, 30), "dipole": (28, 28), "helmholtz": (40, 70), "stokes": (30, 30),
         "stokes_dipole": (45, 45), "blackbox": (20, 20)}


def work(case):
    """Bytes: each coordinate, density and output once.  Operations: those of
    the FMM itself, estimated from the mean number of points in a leaf: pairs
    of neighbouring leaves, points with their leaf's expansion (p terms), and
    the box translations (2 p^2 each)."""
    n, nt, ncut, method, mode = (case[k] for k in ("n", "nt", "ncut", "method", "mode"))
    p = case["p"] ** 2 if method == "blackbox" else case["p"]
    fields = 3 if method.startswith("stokes") else 1
    if case["points"] == "uniform":
        q = n / 4.0 ** max(0, math.ceil(math.log(max(1.0, n / ncut), 4)))
        boxes, near, far = 9, 9 * q, 27
    elif case["points"] == "clusters":
        q = min(n, 0.55 * ncut)
        boxes, near, far = 9, 9 * q, 27
    else:
        q = min(n, 0.7 * ncut)
        boxes, near, far = 3, 3 * q, 9
    if case["targets"] != "self" and case["points"] != "uniform":
        near = near / boxes         # few of the targets have sources beside them
    near = min(near, n)
    nodes = 4.0 / 3.0 * n / q
    small, grad = _PAIR[method]
    translate = fields * nodes * 2.0 * p * p * (far + 9)
    up = small * n * p
    down = small * nt * (p + near)
    inputs = {"dipole": 6, "stokes": 4, "stokes_dipole": 8}.get(method, 3)
    outputs = 3 if fields == 3 else 1
    flops, values = up + translate + down, inputs * n + (2 + outputs) * nt
    if mode == "probe":
        flops, values = grad * nt * (p + near), 5 * nt
    elif mode == "train":
        wide = small if fields == 3 else grad
        flops = 2 * (up + translate) + down + wide * n * (p + near)
        values = inputs * n + 2 * nt + (5 if fields == 3 else 3) * nt + (2 if fields == 3 else 3) * n
    return {"bytes": 8.0 * values, "flops": float(flops)}


# -- the same values by direct sums ------------------------------------------------

# pairs that a direct sum takes within seconds on the GPU
_EXACT_PAIRS = {"laplace": 1e11, "blackbox": 1e11, "dipole": 5e10, "stokes": 5e10,
                "stokes_dipole": 2e10, "helmholtz": 1e10}


def _blocks(tx, ty, x, y, own):
    """(slice, dx, dy, d2, coincident pairs) over the targets; coincident
    pairs have d2 = 1 when a target's own source is left out."""
    step = max(1, 4_000_000 // x.numel())
    for a in range(0, tx.numel(), step):
        k = slice(a, a + step)
        dx, dy = tx[k, None] - x, ty[k, None] - y
        d2 = dx * dx + dy * dy
        same = None
        if own:
            same = d2 == 0.0
            d2.masked_fill_(same, 1.0)
        yield k, dx, dy, d2, same


def _scalar(method, tx, ty, x, y, tau, own, gradient):
    out = torch.empty((3 if gradient else 1, tx.numel()), dtype=torch.float64, device=x.device)
    for k, dx, dy, d2, same in _blocks(tx, ty, x, y, own):
        if method == "helmholtz":
            r = WAVENUMBER * d2.sqrt()
            g = torch.special.modified_bessel_k0(r).div_(TWO_PI)
        else:
            g = torch.log(d2).mul_(-1.0 / FOUR_PI)
        if same is not None:
            g.masked_fill_(same, 0.0)
        out[0, k] = g @ tau
        if gradient:
            if method == "helmholtz":
                h = torch.special.modified_bessel_k1(r).mul_(r).div_(d2).mul_(-1.0 / TWO_PI)
            else:
                h = (-1.0 / TWO_PI) / d2
            out[1, k] = (h * dx) @ tau
            out[2, k] = (h * dy) @ tau
    return out


def _stokes(tx, ty, x, y, f, own):
    out = torch.empty((3, tx.numel()), dtype=torch.float64, device=x.device)
    for k, dx, dy, d2, same in _blocks(tx, ty, x, y, own):
        lg = torch.log(d2).mul_(-0.5)
        inv = 1.0 / d2
        rf = (dx * f[0] + dy * f[1]) * inv
        u = (lg @ f[0] + (dx * rf).sum(1)) / FOUR_PI
        v = (lg @ f[1] + (dy * rf).sum(1)) / FOUR_PI
        q = rf.sum(1) / TWO_PI
        if len(f) > 2:
            w = (dx * f[4] + dy * f[5]) * (dx * f[2] + dy * f[3]) * inv * inv
            if same is not None:
                inv = inv.masked_fill(same, 0.0)
            u = u + (w * dx).sum(1) / math.pi
            v = v + (w * dy).sum(1) / math.pi
            q = q + (2.0 * w.sum(1) - inv @ (f[4] * f[2] + f[5] * f[3])) / math.pi
        out[0, k], out[1, k], out[2, k] = u, v, q
    return out


def exact(case, seed):
    method, mode = case["method"], case["mode"]
    pairs = float(case["n"]) * case["nt"] * (2 if mode == "train" else 1)
    if pairs > _EXACT_PAIRS[method]:
        return None
    s = _inputs(case, seed)
    x, y, tx, ty, own = s["x"], s["y"], s["tx"], s["ty"], case["targets"] == "self"
    if method in ("stokes", "stokes_dipole"):
        u, v, q = _stokes(tx, ty, x, y, s["f"], own)
        if mode != "train":
            return u, v, q
        gu, gv = 2.0 * (u - s["goal"][0]), 2.0 * (v - s["goal"][1])
        fx, fy, _ = _stokes(x, y, tx, ty, [gu, gv], own)
        return u, v, fx, fy
    if method == "dipole":
        out = torch.empty((1, tx.numel()), dtype=torch.float64, device=x.device)
        for k, dx, dy, d2, same in _blocks(tx, ty, x, y, own):
            g = torch.log(d2).mul_(-1.0 / FOUR_PI)
            h = (dx * s["normal"][0] + dy * s["normal"][1]).div_(d2).mul_(1.0 / TWO_PI)
            if same is not None:
                g.masked_fill_(same, 0.0)
                h.masked_fill_(same, 0.0)
            out[0, k] = g @ s["tau"][0] + h @ s["tau"][1]
        return out
    u = _scalar(method, tx, ty, x, y, s["tau"], own, mode == "probe")
    if method == "blackbox":
        return u[0]
    if mode != "train":
        return u
    g = 2.0 * (u[0] - s["goal"])
    v = _scalar(method, x, y, tx, ty, g, own, True)
    return u[0], s["tau"] * v[1], s["tau"] * v[2], v[0]
