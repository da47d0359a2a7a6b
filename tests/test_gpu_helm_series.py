"""Modified Helmholtz near field on each class of series length and across
their edges: direct interactions (one leaf, no expansions) whose q = (k d/2)^2
stays below 1/16, below 1/4, below 1, or straddles all of them and the x > 2
branch, against FP64 direct sums."""
import numpy as np
import pytest

from oracle import direct as odirect
from oracle import kernels as okern
from tests import helpers as H

pytestmark = pytest.mark.gpu


# q <= k^2/2 on the unit square: 0.045, 0.0613, 0.0648, 0.245, 0.259, 0.98, 1.03, 200
@pytest.mark.parametrize("k", [0.3, 0.35, 0.36, 0.7, 0.72, 1.4, 1.44, 20.0])
def test_near_field_series_classes(k):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    ker, _, grad = kernels.modified_helmholtz(k)
    mh, mhg = okern.make_modified_helmholtz(k)[:2]
    x, y, tau = H.uniform(300, 41)
    x[:4], y[:4] = [0, 1, 0, 1], [0, 0, 1, 1]      # the largest distances
    tx, ty, _ = H.uniform(200, 42)
    the_help.clear()
    f = FMM(x, y, ker, 400, 32, bbox=[0, 1, 0, 1])
    f.register_evaluator(grad, grad, "gradient", 3)
    f.build_expansions(tau)
    u = f.target_evaluation(tx, ty)[0]
    g = f.evaluate_to_points(tx, ty, "gradient", False)
    ref = odirect.direct(mh, x, y, tau, tx, ty)[0]
    refg = odirect.direct(mhg, x, y, tau, tx, ty)
    assert H.rel_max_err(u, ref) < 1e-13
    for a, b in zip(g, refg):
        assert H.rel_max_err(a, b) < 1e-12
