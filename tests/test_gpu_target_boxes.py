"""Target location for targets in random order over few boxes, alone and mixed
with boxes that do not repeat: blocks whose targets share every box with
others, none, or some, boxes that meet in the block's slots, and a partly
filled block.  The potentials equal the oracle's and do not depend on the
targets' order."""
import numpy as np
import pytest

from oracle import kernels as okern
from oracle import kifmm2d as okifmm
from tests import helpers as H

pytestmark = pytest.mark.gpu

PARITY_TOL = 1e-12


def _sources(kind):
    if kind == "uniform":
        return *H.uniform(12000, 15)[:2], 30
    if kind == "bitmap":
        return *H.clustered(12000, 4, 0.02, 16)[:2], 30
    return *H.clustered(9000, 3, 1e-5, 17)[:2], 20


@pytest.mark.parametrize("kind", ["uniform", "bitmap", "deep"])
def test_few_boxes_in_random_order(kind):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    x, y, ncut = _sources(kind)
    rng = np.random.default_rng(18)
    tau = rng.standard_normal(x.size)
    the_help.clear()
    f = FMM(x, y, kernels.laplace, ncut, 32, bbox=[0, 1, 0, 1])
    f.build_expansions(tau)
    o = okifmm.FMM(x, y, okern.laplace, ncut, 32, bbox=[0, 1, 0, 1])
    o.build_expansions(tau)
    assert (f.tree.levels > 13) == (kind == "deep")
    tx, ty = [], []
    # `boxes` places that repeat, and a share of the wave's lanes anywhere
    for boxes, single in ((1, 0.0), (2, 0.0), (3, 0.1), (4, 0.5), (5, 0.9), (8, 0.3), (9, 0.0),
                          (12, 0.5), (17, 0.2), (33, 0.0), (64, 0.0), (300, 0.5)):
        cx, cy = rng.random(boxes), rng.random(boxes)
        pick = rng.integers(0, boxes, 512)
        alone = rng.random(512) < single
        tx.append(np.where(alone, rng.random(512), cx[pick]))
        ty.append(np.where(alone, rng.random(512), cy[pick]))
    tx, ty = np.concatenate(tx)[:-7], np.concatenate(ty)[:-7]
    print("boxes", kind, tx.size, "levels", f.tree.levels, flush=True)
    u = f.target_evaluation(tx, ty)[0]
    assert H.rel_max_err(u, o.target_evaluation(tx, ty)[0]) < PARITY_TOL
    p = rng.permutation(tx.size)
    assert H.rel_max_err(f.target_evaluation(tx[p], ty[p])[0], np.asarray(u)[p]) < PARITY_TOL
