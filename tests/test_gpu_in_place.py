"""Outputs that overlap the target coordinates: one and three outputs, x or y
or both inside the output buffer or across its ends, and the evaluation that
allocates nothing; and calls captured into graphs after eager ones.  The same sums per
target as with buffers of their own (the bar is that of two calls of one entry
point)."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu

TOL = 1e-13
NT = 3001


def _plans():
    from flexmm_amd import _lib, kernels
    from flexmm_amd.kifmm2d import FMM, StokesFMM, the_help
    x, y, tau = H.uniform(9000, 81)
    rng = np.random.default_rng(82)
    the_help.clear()
    f = FMM(x, y, kernels.laplace, 30, 32, bbox=[0, 1, 0, 1])
    f.build_expansions(tau)
    s = StokesFMM(x, y, 32, 30, bbox=[0, 1, 0, 1])
    s.build_expansions(tau, rng.standard_normal(x.size))
    return {"potential": (f, _lib.EVAL_POTENTIAL, 1), "gradient": (f, _lib.EVAL_GRADIENT, 3),
            "stokes": (s, _lib.EVAL_STOKES, 3)}


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("what", ["potential", "gradient", "stokes"])
@pytest.mark.parametrize("place", ["x_first", "y_last", "both", "across_begin", "across_end"])
def test_output_over_the_targets(what, place, noalloc):
    import torch
    from flexmm_amd import _lib
    f, ev, nout = _plans()[what]
    call = f.lib.fmm2d_evaluate_noalloc if noalloc else f.lib.fmm2d_evaluate
    tx, ty = (torch.from_numpy(a).cuda() for a in H.uniform(NT, 83)[:2])
    print("in place", what, place, noalloc, flush=True)

    def run(px, py, out):
        _lib.check(call(f.handle, px.data_ptr(), py.data_ptr(), NT, ev, 0, out.data_ptr(), None))
        torch.cuda.synchronize()
        return out.cpu().numpy().reshape(nout, NT)
    torch.cuda.synchronize()
    ref = run(tx, ty, torch.empty(nout * NT, dtype=torch.float64, device="cuda"))
    # out = buf[NT : NT + nout NT], the coordinates moved to offsets in buf
    buf = torch.full(((nout + 2) * NT,), float("nan"), dtype=torch.float64, device="cuda")
    out = buf[NT:NT + nout * NT]
    at = {"x_first": (NT, None), "y_last": (None, nout * NT),
          "both": (NT, 2 * NT), "across_begin": (NT - 700, None),
          "across_end": (None, NT + nout * NT - 700)}[place]
    if place == "both" and nout == 1:
        at = (NT - 1500, NT + 1501)   # disjoint, each half inside the output
    px, py = (c if o is None else buf[o:o + NT].copy_(c) for c, o in zip((tx, ty), at))
    torch.cuda.synchronize()
    got = run(px, py, out)
    for k in range(nout):
        assert H.rel_max_err(got[k], ref[k]) < TOL


@pytest.mark.parametrize("what", ["potential", "gradient", "stokes"])
def test_capture_after_a_call_with_separate_buffers(what):
    """A call that allocated for NT targets is enough for a captured call over
    its targets; every replay gives the eager result."""
    import torch
    from flexmm_amd import _lib
    f, ev, nout = _plans()[what]
    tx, ty = (torch.from_numpy(a).cuda() for a in H.uniform(NT, 84)[:2])
    ref = torch.empty(nout * NT, dtype=torch.float64, device="cuda")
    buf = torch.empty(max(2, nout) * NT, dtype=torch.float64, device="cuda")
    print("capture in place", what, flush=True)

    def call(px, py, out):
        _lib.check(f.lib.fmm2d_evaluate(f.handle, px.data_ptr(), py.data_ptr(), NT, ev, 0,
                                        out.data_ptr(),
                                        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    call(tx, ty, ref)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(buf[:NT], buf[NT:2 * NT], buf)
    for _ in range(3):
        buf[:NT].copy_(tx)
        buf[NT:2 * NT].copy_(ty)
        graph.replay()
        torch.cuda.synchronize()
        got = buf[:nout * NT].cpu().numpy().reshape(nout, NT)
        for k, r in enumerate(ref.cpu().numpy().reshape(nout, NT)):
            assert H.rel_max_err(got[k], r) < TOL
        call(tx, ty, ref)   # the program's own work between the replays
        torch.cuda.synchronize()


def test_capture_on_a_smaller_tree():
    """The scratch of an evaluation on a larger tree is enough on a smaller one
    (whose few boxes take several counters each)."""
    import torch
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    from flexmm_amd.kifmm2d import fmm as module
    module._plan_pool.clear()
    the_help.clear()
    tx, ty = (torch.from_numpy(a).cuda() for a in H.uniform(NT, 85)[:2])
    out = torch.empty(NT, dtype=torch.float64, device="cuda")
    f = None
    for n in (40000, 9000):
        x, y, tau = (torch.from_numpy(a).cuda() for a in H.uniform(n, 86))
        if f is not None:
            handle = f.handle.value
            f.close()
        f = FMM(x, y, kernels.laplace, 6, 32, bbox=[0, 1, 0, 1])
        f.build_expansions(tau)
        print("boxes", f.tree.n_leaves, flush=True)
        torch.cuda.synchronize()

        def call():
            from flexmm_amd import _lib
            _lib.check(f.lib.fmm2d_evaluate(f.handle, tx.data_ptr(), ty.data_ptr(), NT,
                                            _lib.EVAL_POTENTIAL, 0, out.data_ptr(),
                                            torch.cuda.current_stream().cuda_stream))
        if n == 40000:
            assert f.tree.n_leaves > 4096
            call()
    assert f.handle.value == handle and 512 < f.tree.n_leaves <= 4096
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    got = []
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        got.append(out.cpu().numpy())
        call()
        torch.cuda.synchronize()
        ref = out.cpu().numpy()
    for g in got:
        assert H.rel_max_err(g, ref) < TOL
