"""Device memory that a plan takes for its operators (include/flexmm_amd.h,
fmm2d_set_operators): room for 32 levels of the operator blocks and of the
kernels' own copy, which leaves the M2L blocks out where no kernel reads them."""
import pytest

pytestmark = pytest.mark.gpu

SLACK = 6 << 20   # two allocations rounded up to 2 MiB, and the copy's queue


@pytest.mark.parametrize("p", [32, 48, 64])
@pytest.mark.parametrize("kernel,precision,blocks", [
    ("laplace", "fp64", 50), ("laplace", "mixed", 10), ("helmholtz", "mixed_m2l", 10),
    ("stokes", "mixed", 50)])
def test_operator_memory(p, kernel, precision, blocks):
    import torch
    from flexmm_amd import _lib, kernels
    from flexmm_amd.kifmm2d.fmm import _PRECISIONS, _Plan
    lib = _lib.load()
    ker = {"laplace": kernels.laplace, "helmholtz": kernels.modified_helmholtz(3.0)[0],
           "stokes": kernels.stokeslet}[kernel]
    n = lib.fmm2d_operator_size(p)
    ops = torch.zeros(n, dtype=torch.float64, device="cuda")
    pe = -(-p // 16) * 16
    print("operator memory", kernel, precision, p, flush=True)
    plan = _Plan(lib, ker, p, _PRECISIONS[precision])
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    _lib.check(lib.fmm2d_set_operators(plan.h, 2, ops.data_ptr(), n, None))
    torch.cuda.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    plan.close()
    assert used <= 32 * 8 * (n + blocks * pe * pe) + SLACK
