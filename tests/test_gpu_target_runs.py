"""Target location by the order of the targets: runs of equal boxes that fill
a wave in every way the grouping tells apart (few runs, one more than the
limit of the joined form, two lanes each, one each, a box that comes back), in
complete trees, trees with the bitmap index and deeper ones.  The potentials
equal the oracle's and do not depend on the targets' order."""
import numpy as np
import pytest

from oracle import kernels as okern
from oracle import kifmm2d as okifmm
from tests import helpers as H

pytestmark = pytest.mark.gpu

PARITY_TOL = 1e-12


def _sources(kind):
    if kind == "complete":
        return *H.uniform(20000, 5)[:2], 30
    if kind == "bitmap":
        return *H.clustered(20000, 4, 0.02, 6)[:2], 30
    return *H.clustered(12000, 3, 1e-5, 7)[:2], 20


@pytest.mark.parametrize("kind", ["complete", "bitmap", "deep"])
def test_runs_of_targets(kind):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y, ncut = _sources(kind)
    rng = np.random.default_rng(8)
    tau = rng.standard_normal(x.size)
    the_help.clear()
    f = FMM(x, y, kernels.laplace, ncut, 32, bbox=[0, 1, 0, 1])
    f.build_expansions(tau)
    o = okifmm.FMM(x, y, okern.laplace, ncut, 32, bbox=[0, 1, 0, 1])
    o.build_expansions(tau)
    assert (f.tree.levels > 13) == (kind == "deep")
    # run lengths that give 4, 15, 16, 17, 32 and 64 runs per wave, around
    # places that lie in different boxes, then every box twice in one wave
    tx, ty = [], []
    for length in (16, 5, 4, 3, 2, 1):
        n = 320 // length
        cx, cy = rng.random(n), rng.random(n)
        tx.append(np.repeat(cx, length))
        ty.append(np.repeat(cy, length))
    cx, cy = rng.random(32), rng.random(32)
    tx.append(np.tile(cx, 2))
    ty.append(np.tile(cy, 2))
    tx, ty = np.concatenate(tx)[:-3], np.concatenate(ty)[:-3]
    print("runs", kind, tx.size, "levels", f.tree.levels, flush=True)
    u = f.target_evaluation(tx, ty)[0]
    assert H.rel_max_err(u, o.target_evaluation(tx, ty)[0]) < PARITY_TOL
    p = rng.permutation(tx.size)
    assert H.rel_max_err(f.target_evaluation(tx[p], ty[p])[0], np.asarray(u)[p]) < PARITY_TOL
