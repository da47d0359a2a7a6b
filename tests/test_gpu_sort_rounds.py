"""Key sort rounds of many segments: more than 512 depth-8 cells go on to the
third radix round, all short (several segments per block), exactly at the
line, or with one that spans more than 16 chunks of 4096 points (a block per
segment).  The permutation holds every point once and the tree is the
oracle's."""
import numpy as np
import pytest

from oracle import tree as otree
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,dense", [(512, 0), (513, 0), (515, 9000), (900, 0), (900, 70000)])
def test_rounds_of_many_segments(cells, dense):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    rng = np.random.default_rng([cells, dense])
    w = 1 / 256
    ids = rng.permutation(256 * 256)[:cells]
    cx, cy = (ids // 256) * w, (ids % 256) * w
    per = rng.integers(25, 90, cells)        # all over the leaf capacity
    x, y = np.repeat(cx, per), np.repeat(cy, per)
    x, y = x + w * rng.uniform(0.01, 0.99, x.size), y + w * rng.uniform(0.01, 0.99, x.size)
    if dense:
        x = np.concatenate([x, cx[0] + w * rng.uniform(0.01, 0.99, dense)])
        y = np.concatenate([y, cy[0] + w * rng.uniform(0.01, 0.99, dense)])
    p = rng.permutation(x.size)
    x, y = x[p].copy(), y[p].copy()
    print("cells", cells, "dense", dense, "n", x.size, flush=True)
    the_help.clear()
    f = FMM(x, y, kernels.laplace, 20, 16, bbox=[0, 1, 0, 1])
    perm = f.tree_array("perm").cpu().numpy().astype(np.int64)
    assert np.array_equal(np.sort(perm), np.arange(x.size))
    assert np.array_equal(f.tree_array("sx").cpu().numpy(), x[perm])
    ora = otree.Tree(x, y, 20, f.bbox)
    assert H.compare_trees_fast(f, ora) == sum(l.n_node for l in ora.Levels)
