"""Modified Helmholtz evaluations around the box width past which the near
field takes the full series only (one wave per item: a tree of more than 16384
evaluation boxes), potential and gradient against FP64 direct sums, and the
reference's self-exclusion."""
import numpy as np
import pytest

from oracle import direct as odirect
from oracle import kernels as okern
from tests import helpers as H

pytestmark = pytest.mark.gpu


# leaves of width 1/256: k w = 0.39, 0.41, 0.59, 0.61, 1.2
@pytest.mark.parametrize("k", [100.0, 105.0, 151.0, 156.0, 300.0])
def test_full_series_of_wide_boxes(k):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    m = 256
    rng = np.random.default_rng(51)
    g = np.stack(np.meshgrid(np.arange(m), np.arange(m), indexing="ij"), -1).reshape(-1, 2)
    pts = (g + rng.uniform(0.1, 0.9, (m * m, 2))) / m
    x, y, tau = pts[:, 0].copy(), pts[:, 1].copy(), rng.standard_normal(m * m)
    ker, _, grad = kernels.modified_helmholtz(k)
    mh, mhg = okern.make_modified_helmholtz(k)[:2]
    the_help.clear()
    f = FMM(x, y, ker, 1, 60, bbox=[0, 1, 0, 1])
    assert f.tree.widths[-1] == 1 / m and f.tree.n_leaves > 16384
    f.register_evaluator(grad, grad, "gradient", 3)
    f.build_expansions(tau)
    print("wide boxes", k / m, flush=True)
    tx, ty, _ = H.uniform(400, 52)
    u = f.target_evaluation(tx, ty)[0]
    assert H.rel_max_err(u, odirect.direct(mh, x, y, tau, tx, ty)[0]) < 1e-12
    got = f.evaluate_to_points(tx, ty, "gradient", False)
    for a, b in zip(got, odirect.direct(mhg, x, y, tau, tx, ty)):
        assert H.rel_max_err(a, b) < 1e-11   # ten times the potential's, as elsewhere
    sel = np.arange(0, x.size, 331)
    us = f.source_evaluation(x, y)[0][sel]
    assert H.rel_max_err(us, odirect.direct(mh, x, y, tau, x[sel], y[sel], check=True)[0]) < 1e-12
