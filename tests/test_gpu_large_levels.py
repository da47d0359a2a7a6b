"""A tree of more than 16384 S2M boxes whose two deepest levels have more than
4096 nodes, half of the last level's fake: a leaf's sources are summed by one
wave, and large levels run the wave-per-16-boxes kernels, the downward one in
the tree's column order.  All source kinds, and every padding of p, against
the oracle, direct sums, or (mixed precision) the FP64 form."""
import numpy as np
import pytest

from oracle import direct as odirect
from oracle import kernels as okern
from oracle import kifmm2d as okifmm
from tests import helpers as H

pytestmark = pytest.mark.gpu

PARITY_TOL = 1e-12
MIXED_TOL = 1e-7   # the mixed form's bar against FP64
BOX = [0, 1, 0, 1]


def _points(seed=9, m=128):
    """m x m cells, half of them with one point per quadrant, the others with
    one (leaf capacity 1)."""
    rng = np.random.default_rng(seed)
    four = rng.random((m, m)) < 0.5
    i, j = np.nonzero(~four)
    pts = [np.stack([i, j], 1) + rng.uniform(0.1, 0.9, (i.size, 2))]
    i, j = np.nonzero(four)
    for a in (0.0, 0.5):
        for b in (0.0, 0.5):
            pts.append(np.stack([i + a, j + b], 1) + rng.uniform(0.05, 0.45, (i.size, 2)))
    p = np.concatenate(pts)
    p = p[rng.permutation(len(p))] / m
    return p[:, 0].copy(), p[:, 1].copy()


def _targets():
    rng = np.random.default_rng(10)
    return rng.random(700), rng.random(700)


def _check_tree(t):
    assert t.n_s2m > 16384 and min(t.level_nodes[-2:]) > 4096
    assert t.level_nodes[-1] != 4 ** (t.levels - 1)


@pytest.mark.parametrize("p", [13, 16, 30, 32, 41, 48, 60])
def test_laplace(p):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y = _points()
    tx, ty = _targets()
    tau = np.random.default_rng(11).standard_normal(x.size)
    print("large levels p", p, flush=True)
    the_help.clear()
    f = FMM(x, y, kernels.laplace, 1, p, bbox=BOX)
    _check_tree(f.tree)
    f.build_expansions(tau)
    o = okifmm.FMM(x, y, okern.laplace, 1, p, bbox=BOX)
    o.build_expansions(tau)
    assert H.rel_max_err(f.target_evaluation(tx, ty)[0], o.target_evaluation(tx, ty)[0]) < PARITY_TOL


def test_dipole():
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y = _points()
    tx, ty = _targets()
    rng = np.random.default_rng(12)
    tau, th = rng.standard_normal((2, x.size)), rng.uniform(0, 2 * np.pi, x.size)
    dv = np.stack([np.cos(th), np.sin(th)])
    the_help.clear()
    f = FMM(x, y, kernels.laplace, 1, 32, bbox=BOX)
    _check_tree(f.tree)
    f.register_upwardor(kernels.laplace_slp_dlp, "slp+dlp")
    f.register_evaluator(f.helper.functions["kernel_app"], kernels.laplace_slp_dlp, "slp+dlp->u", 1)
    f.build_expansions(tau, "slp+dlp", dv)
    o = okifmm.FMM(x, y, okern.laplace, 1, 32, bbox=BOX)
    o.register_evaluator(lambda *a: (okern.laplace(*a),), "slp+dlp->u", 1, src=okern.laplace_slp_dlp)
    o.build_expansions(tau, okern.laplace_slp_dlp, dv)
    u = f.evaluate_to_points(tx, ty, "slp+dlp->u", False)[0]
    assert H.rel_max_err(u, o.evaluate_to_points(tx, ty, "slp+dlp->u", False)[0]) < PARITY_TOL


def test_helmholtz():
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y = _points()
    tx, ty = _targets()
    tau = np.random.default_rng(13).standard_normal(x.size)
    the_help.clear()
    f = FMM(x, y, kernels.modified_helmholtz(20.0)[0], 1, 32, bbox=BOX)
    _check_tree(f.tree)
    f.build_expansions(tau)
    mh, _ = okern.make_modified_helmholtz(20.0)
    o = okifmm.FMM(x, y, mh, 1, 32, bbox=BOX)
    o.build_expansions(tau)
    assert H.rel_max_err(f.target_evaluation(tx, ty)[0], o.target_evaluation(tx, ty)[0]) < PARITY_TOL


@pytest.mark.parametrize("dipole", [False, True])
def test_stokes(dipole):
    from flexmm_amd.kifmm2d import StokesFMM, the_help
    x, y = _points()
    tx, ty = _targets()
    rng = np.random.default_rng(14)
    fx, fy, gx, gy = rng.standard_normal((4, x.size))
    th = rng.uniform(0, 2 * np.pi, x.size)
    nx, ny = np.cos(th), np.sin(th)
    the_help.clear()
    f = StokesFMM(x, y, 64, 1, bbox=BOX)
    _check_tree(f.tree)
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


@pytest.mark.parametrize("p", [12, 24, 32, 40, 48])
def test_mixed_laplace_keeps_its_bar(p):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y = _points()
    tx, ty = _targets()
    tau = np.random.default_rng(15).standard_normal(x.size)
    the_help.clear()
    u = []
    for precision in ("fp64", "mixed"):
        print("large levels", precision, p, flush=True)
        f = FMM(x, y, kernels.laplace, 1, p, bbox=BOX, precision=precision)
        _check_tree(f.tree)
        f.build_expansions(tau)
        u.append(f.target_evaluation(tx, ty)[0])
    assert H.rel_max_err(u[1], u[0]) < MIXED_TOL


@pytest.mark.parametrize("p", [20, 32, 48])
def test_mixed_stokes_keeps_its_bar(p):
    from flexmm_amd.kifmm2d import StokesFMM, the_help
    x, y = _points()
    tx, ty = _targets()
    fx, fy = np.random.default_rng(16).standard_normal((2, x.size))
    the_help.clear()
    got = []
    for precision in ("fp64", "mixed"):
        print("large levels Stokes", precision, p, flush=True)
        f = StokesFMM(x, y, p, 1, bbox=BOX, precision=precision)
        _check_tree(f.tree)
        f.build_expansions(fx, fy)
        got.append(f.evaluate_to_points(tx, ty, False))
    for a, b in zip(got[1], got[0]):
        assert H.rel_max_err(np.asarray(a), np.asarray(b)) < MIXED_TOL
