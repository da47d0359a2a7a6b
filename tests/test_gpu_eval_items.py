"""Evaluation items at their edges: leaves with every number of targets around
the few-target, full-wave and two-item limits, colleagues with fewer sources
than an item has waves, for items shared by the waves of a block (few boxes)
and one wave per item (many boxes), against the oracle and direct sums."""
import numpy as np
import pytest

from oracle import direct as odirect
from oracle import kernels as okern
from oracle import kifmm2d as okifmm
from tests import helpers as H

pytestmark = pytest.mark.gpu

PARITY_TOL = 1e-12
COUNTS = [0, 1, 2, 3, 4, 5, 7, 8, 9, 15, 17, 31, 32, 33, 47, 63, 64, 65, 96, 97, 128, 130]


def _grid_sources(m, rng, per):
    i, j = np.meshgrid(np.arange(m), np.arange(m), indexing="ij")
    i, j = np.repeat(i.ravel(), per), np.repeat(j.ravel(), per)
    return (i + rng.uniform(0.05, 0.95, i.size)) / m, (j + rng.uniform(0.05, 0.95, j.size)) / m


def _problem(many):
    """Sources of a complete tree (128 x 128 leaves of one source, or 8 x 8
    leaves of three) and targets with COUNTS[k] of them in the k-th of a row
    of its leaves."""
    rng = np.random.default_rng(31)
    m, per, ncut = (128, 1, 1) if many else (8, 3, 3)
    x, y = _grid_sources(m, rng, per)
    tx, ty = [], []
    for k, c in enumerate(COUNTS):
        ci, cj = (k % 7, k // 7) if not many else (5 * k, 100)
        tx.append((ci + rng.uniform(0.02, 0.98, c)) / m)
        ty.append((cj + rng.uniform(0.02, 0.98, c)) / m)
    return x, y, ncut, np.concatenate(tx), np.concatenate(ty), rng


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("p", [13, 60])
def test_laplace_items(many, p):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y, ncut, tx, ty, rng = _problem(many)
    tau = rng.standard_normal(x.size)
    print("many", many, "p", p, flush=True)
    the_help.clear()
    f = FMM(x, y, kernels.laplace, ncut, p, bbox=[0, 1, 0, 1])
    f.register_evaluator(kernels.laplace_gradient, kernels.laplace_gradient, "gradient", 3)
    f.build_expansions(tau)
    o = okifmm.FMM(x, y, okern.laplace, ncut, p, bbox=[0, 1, 0, 1])
    o.register_evaluator(okern.laplace_gradient, "gradient", 3)
    o.build_expansions(tau)
    assert H.rel_max_err(f.target_evaluation(tx, ty)[0], o.target_evaluation(tx, ty)[0]) < PARITY_TOL
    g, go = f.evaluate_to_points(tx, ty, "gradient", False), o.evaluate_to_points(tx, ty, "gradient", False)
    for k in range(3):
        assert H.rel_max_err(g[k], go[k]) < 10 * PARITY_TOL
    # a target on a source: +inf without self-exclusion, excluded with it
    tx[-1], ty[-1] = x[0], y[0]
    u = f.target_evaluation(tx, ty)[0]
    assert u[-1] == np.inf and np.isfinite(u[:-1]).all()
    us, uo = f.source_evaluation(tx, ty)[0], o.source_evaluation(tx, ty)[0]
    assert H.rel_max_err(us, uo) < PARITY_TOL


@pytest.mark.parametrize("many", [False, True])
def test_dipole_items(many):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y, ncut, tx, ty, rng = _problem(many)
    tau = rng.standard_normal((2, x.size))
    th = rng.uniform(0, 2 * np.pi, x.size)
    dv = np.stack([np.cos(th), np.sin(th)])
    the_help.clear()
    f = FMM(x, y, kernels.laplace, ncut, 32, bbox=[0, 1, 0, 1])
    f.register_upwardor(kernels.laplace_slp_dlp, "slp+dlp")
    f.register_evaluator(f.helper.functions["kernel_app"], kernels.laplace_slp_dlp, "slp+dlp->u", 1)
    f.build_expansions(tau, "slp+dlp", dv)
    o = okifmm.FMM(x, y, okern.laplace, ncut, 32, bbox=[0, 1, 0, 1])
    o.register_evaluator(lambda *a: (okern.laplace(*a),), "slp+dlp->u", 1, src=okern.laplace_slp_dlp)
    o.build_expansions(tau, okern.laplace_slp_dlp, dv)
    u = f.evaluate_to_points(tx, ty, "slp+dlp->u", False)[0]
    uo = o.evaluate_to_points(tx, ty, "slp+dlp->u", False)[0]
    assert H.rel_max_err(u, uo) < PARITY_TOL


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("dipole", [False, True])
def test_stokes_items(many, dipole):
    from flexmm_amd.kifmm2d import StokesFMM
    x, y, ncut, tx, ty, rng = _problem(many)
    fx, fy, gx, gy = rng.standard_normal((4, x.size))
    th = rng.uniform(0, 2 * np.pi, x.size)
    nx, ny = np.cos(th), np.sin(th)
    f = StokesFMM(x, y, 64, ncut, bbox=[0, 1, 0, 1])
    if dipole:
        f.build_expansions_dipole(fx, fy, gx, gy, nx, ny)
        got = f.evaluate_to_points_dipole(tx, ty, False)
        ref = odirect.direct_stokes_dipole(x, y, fx, fy, gx, gy, nx, ny, tx, ty)
    else:
        f.build_expansions(fx, fy)
        got = f.evaluate_to_points(tx, ty, False)
        ref = odirect.direct_stokes(x, y, fx, fy, tx, ty)
    for a, b in zip(got, ref):
        assert H.rel_max_err(np.asarray(a), b) < 5e-11   # the p = 64 bar of the Stokes tests


def test_output_over_the_targets():
    """An output buffer that overlaps the target coordinates."""
    import torch
    from flexmm_amd import _lib, kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y, ncut, tx, ty, rng = _problem(False)
    the_help.clear()
    f = FMM(x, y, kernels.laplace, ncut, 32, bbox=[0, 1, 0, 1])
    f.build_expansions(rng.standard_normal(x.size))
    u = f.target_evaluation(tx, ty)[0]
    dx = torch.tensor(tx, device=f.device)
    dy = torch.tensor(ty, device=f.device)
    torch.cuda.synchronize()
    s = torch.cuda.current_stream().cuda_stream
    _lib.check(f.lib.fmm2d_evaluate(f.handle, dx.data_ptr(), dy.data_ptr(), dx.numel(),
                                    _lib.EVAL_POTENTIAL, 0, dx.data_ptr(), s))
    assert np.array_equal(dx.cpu().numpy(), u) or H.rel_max_err(dx.cpu().numpy(), u) < 1e-14
