"""Trees by their number of levels.  Trees of up to 13 levels keep their split
cells as bitmaps, deeper ones as sorted code lists: both against the oracle
tree (canonical comparison, centres bit for bit) for every depth around the
places where the bitmap kernels change their form, and the node lists of a
tree with more nodes than one pass of block sums takes against cumulative sums
of its flags."""
import numpy as np
import pytest

from oracle import tree as otree
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _build(x, y, ncut):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    the_help.clear()
    return FMM(x, y, kernels.laplace, ncut, 16, bbox=[0, 1, 0, 1])


def _with_cells(k, seed, nbg=200):
    """Background points and, in two cells of depth k (one in the domain's
    corner), nine points spread over the cell's quadrants: depth k splits and
    no deeper one (leaf capacity 8)."""
    rng = np.random.default_rng(seed)
    x, y = rng.random(nbg), rng.random(nbg)
    w = 2.0 ** -k
    q = np.arange(9) % 4
    for cx, cy in ((np.floor(0.3 / w) * w, np.floor(0.7 / w) * w), (1 - w, 0.0)):
        x = np.concatenate([x, cx + w * (0.5 * (q % 2) + 0.05 + 0.4 * rng.random(9))])
        y = np.concatenate([y, cy + w * (0.5 * (q // 2) + 0.05 + 0.4 * rng.random(9))])
    return x, y


@pytest.mark.parametrize("k", range(1, 16))
def test_levels_match_oracle(k):
    x, y = _with_cells(k, 500 + k)
    print("depth", k, flush=True)
    f = _build(x, y, 8)
    if k >= 6:
        assert f.tree.levels == k + 2
    ora = otree.Tree(x, y, 8, f.bbox)
    n = H.compare_canonical(H.gpu_canonical(f), ora.canonical())
    assert n == sum(l.n_node for l in ora.Levels)


@pytest.mark.parametrize("n,ncut", [(1, 8), (8, 8), (9, 8), (40, 3)])
def test_shallow_trees_match_oracle(n, ncut):
    rng = np.random.default_rng(n)
    x, y = rng.random(n), rng.random(n) ** 3
    f = _build(x, y, ncut)
    ora = otree.Tree(x, y, ncut, f.bbox)
    H.compare_canonical(H.gpu_canonical(f), ora.canonical())


@pytest.mark.parametrize("kind", ["jittered_grid_with_hole", "tight_clusters"])
def test_node_lists_of_many_nodes(kind):
    rng = np.random.default_rng(9)
    if kind == "tight_clusters":
        c = rng.uniform(0.2, 0.8, (4, 2))
        p = c[rng.integers(0, 4, 900_000)] + 3e-5 * rng.standard_normal((900_000, 2))
        ncut = 2
    else:
        g = np.stack(np.meshgrid(np.arange(1024), np.arange(1024), indexing="ij"), -1)
        p = (g.reshape(-1, 2) + rng.uniform(0.1, 0.9, (1024 * 1024, 2))) / 1024
        p = p[np.hypot(p[:, 0] - 0.3, p[:, 1] - 0.6) > 0.1]
        p = p[rng.permutation(len(p))]
        ncut = 1
    print("many nodes", kind, flush=True)
    f = _build(p[:, 0].copy(), p[:, 1].copy(), ncut)
    assert (f.tree.levels <= 13) == (kind != "tight_clusters")
    a = {k: f.tree_array(k).cpu().numpy() for k in ("flags", "evalid", "row", "level", "bot", "top",
                                                    "child", "parent")}
    fl, lev = a["flags"], a["level"]
    assert fl.size > 64 * 8192
    leaf = (fl & 1) != 0
    assert np.array_equal(a["evalid"], np.where(leaf, np.cumsum(leaf) - 1, -1))
    assert f.tree.n_leaves == leaf.sum()
    g0 = int((lev < 2).sum())
    grp = ((fl[g0:].reshape(-1, 4) & 64) != 0).any(axis=1)
    row = np.where(grp, 4 * (np.cumsum(grp) - 1), -1)[:, None] + np.arange(4) * grp[:, None]
    assert np.array_equal(a["row"][g0:], row.ravel()) and np.all(a["row"][:g0] == -1)
    assert f.tree.n_rows == 4 * grp.sum()
    assert f.tree.n_s2m == ((fl[g0:] & 8) != 0).sum()
    for d in range(2, f.tree.levels):
        assert f.tree.row_off[d] == (a["row"][(lev < d)] >= 0).sum()
    # a node's children cut its point range into four
    par = np.flatnonzero(a["child"] >= 0)
    ch = a["child"][par]
    assert np.array_equal(a["bot"][ch], a["bot"][par])
    assert np.array_equal(a["top"][ch + 3], a["top"][par])
    for j in range(3):
        assert np.array_equal(a["top"][ch + j], a["bot"][ch + j + 1])
    assert np.array_equal(a["parent"][ch], par)
