"""The dense FP64 M2L at its edges, against the oracle at the FP64 parity bar:
every padding of the operator (p rounded up to 16, an odd or even number of
k-steps) in each shape of the kernel (two blocks per tile on small trees, one
column group on adaptive and mid-sized trees, two on large complete trees with
a remainder of groups in the last tile)."""
import numpy as np
import pytest

from oracle import kernels as okern
from oracle import kifmm2d as okifmm
from tests import helpers as H

pytestmark = pytest.mark.gpu

PARITY_TOL = 1e-12


def _points(kind):
    rng = np.random.default_rng(17)
    if kind == "small":          # 5 complete levels: under 512 tiles
        return rng.random(3000), rng.random(3000), 20
    if kind == "adaptive":       # a curve: adaptive, over 512 tiles
        th = rng.uniform(0, 2 * np.pi, 9000)
        return 0.5 + 0.4 * np.cos(th), 0.5 + 0.4 * np.sin(th), 6
    # one point per cell of a 128 x 128 grid: a complete tree of 8 levels
    i, j = np.meshgrid(np.arange(128), np.arange(128), indexing="ij")
    x = (i.ravel() + rng.uniform(0.1, 0.9, 128 * 128)) / 128
    y = (j.ravel() + rng.uniform(0.1, 0.9, 128 * 128)) / 128
    return x, y, 1


@pytest.mark.parametrize("kind,p", [("small", 4), ("small", 16), ("small", 20), ("small", 32),
                                    ("small", 36), ("small", 48), ("small", 57), ("small", 60),
                                    ("small", 64), ("adaptive", 13), ("adaptive", 28),
                                    ("adaptive", 48), ("adaptive", 60), ("complete", 16),
                                    ("complete", 27), ("complete", 44), ("complete", 60),
                                    ("complete", 63)])
def test_dense_m2l_shapes(kind, p):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y, ncut = _points(kind)
    rng = np.random.default_rng(18)
    tau = rng.standard_normal(x.size)
    tx, ty = rng.random(500), rng.random(500)
    print(kind, "p", p, flush=True)
    the_help.clear()
    f = FMM(x, y, kernels.laplace, ncut, p, bbox=[0, 1, 0, 1])
    f.build_expansions(tau)
    u = f.target_evaluation(tx, ty)[0]
    o = okifmm.FMM(x, y, okern.laplace, ncut, p, bbox=[0, 1, 0, 1])
    o.build_expansions(tau)
    uo = o.target_evaluation(tx, ty)[0]
    err = H.rel_max_err(u, uo)
    print("levels", f.tree.levels, "nodes", f.tree.n_nodes, "err %.2e" % err)
    assert err < PARITY_TOL
