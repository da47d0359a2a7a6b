"""The mixed Stokeslet M2L by its number of 16-box tiles: blocks that take one,
two or all row blocks of a tile, at both padded sizes and with padding inside
the last row block, against the FP64 form."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

MIXED_TOL = 1e-7   # the mixed form's bar against FP64


def _tiles(t):
    return sum(4 * -(-(k // 4) // 16) for k in t.level_nodes[2:])


# uniform points: 4, 24 and 344 tiles; clusters between
@pytest.mark.parametrize("p", [20, 32, 50, 64])
@pytest.mark.parametrize("n,ncut,lo,hi", [(1000, 100, 1, 64), (4000, 50, 1, 64),
                                          (16000, 60, 65, 128), (40000, 30, 129, 10 ** 6)])
def test_row_splits(n, ncut, lo, hi, p):
    from flexmm_amd.kifmm2d import StokesFMM, the_help
    x, y, fx = H.uniform(n, 61)
    fy = np.random.default_rng(62).standard_normal(n)
    tx, ty, _ = H.uniform(500, 63)
    the_help.clear()
    got = []
    for precision in ("fp64", "mixed"):
        f = StokesFMM(x, y, p, ncut, bbox=[0, 1, 0, 1], precision=precision)
        print("tiles", _tiles(f.tree), precision, p, flush=True)
        assert lo <= _tiles(f.tree) <= hi
        f.build_expansions(fx, fy)
        got.append(f.evaluate_to_points(tx, ty, False))
    for a, b in zip(got[1], got[0]):
        assert H.rel_max_err(np.asarray(a), np.asarray(b)) < MIXED_TOL
