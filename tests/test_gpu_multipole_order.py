"""The order of the sums that lead to a multipole.  The pseudo-inverse
amplifies the rounding of the check potentials (6e-7 of a multipole at p 64),
which cancels again in FP64, but the FP32 M2L rounds the multipoles in
between: another order of summation draws that rounding error anew.  Multipoles
of mixed plans are therefore functions of the sorted points alone, whatever the
size of the problem: level products of large levels are ascending chains of
FMAs, emulated here bit for bit, and a leaf's S2M does not depend on how many
leaves there are."""
import ctypes
import ctypes.util

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL_LEVEL_ROWS = 4096   # larger levels run the wave-per-16-boxes kernel
SPLIT_LEAVES = 16384      # S2M boxes up to which FP64 plans share a leaf among four waves


def _chain(A, b, acc):
    """acc + A b as one FMA per entry, columns in ascending order (zero columns
    leave the sum as it is)."""
    fma = ctypes.CDLL(ctypes.util.find_library("m")).fma
    fma.restype = ctypes.c_double
    fma.argtypes = [ctypes.c_double] * 3
    out = []
    for r in range(A.shape[0]):
        s = float(acc[r])
        for k in range(A.shape[1]):
            s = fma(float(A[r, k]), float(b[k]), s)
        out.append(s)
    return np.array(out)


@pytest.mark.parametrize("precision,p", [("mixed", 64), ("mixed", 60), ("mixed", 40), ("mixed", 32),
                                         ("mixed", 16), ("mixed_m2l", 60)])
def test_large_level_products_are_ascending_fma_chains(precision, p):
    from flexmm_amd import kernels
    from flexmm_amd.kifmm2d import FMM, the_help
    the_help.clear()   # cached widths would snap the box
    m = 256   # one point per cell of depth 8
    rng = np.random.default_rng(3)
    g = np.stack(np.meshgrid(np.arange(m), np.arange(m), indexing="ij"), -1).reshape(-1, 2)
    pts = (g + rng.uniform(0.2, 0.8, (m * m, 2))) / m
    print("large level", precision, p, flush=True)
    f = FMM(pts[:, 0].copy(), pts[:, 1].copy(), kernels.laplace, 1, p, bbox=[0, 1, 0, 1],
            precision=precision)
    f.build_expansions(rng.standard_normal(m * m))
    t, d = f.tree, 7
    assert t.row_off[d + 1] - t.row_off[d] > SMALL_LEVEL_ROWS
    mult = f.expansion_array("multipole").cpu().numpy().reshape(-1, t.PD)
    row, child, level = (f.tree_array(k).cpu().numpy() for k in ("row", "child", "level"))
    ops = f.helper.device_operators(t.widths[d], f.device).cpu().numpy()
    blocks = ops[:50 * t.PD * t.PD].reshape(50, t.PD, t.PD)[:, :p, :p]
    nodes = np.flatnonzero(level == d)
    for g in nodes[[0, 1, 63, 64, nodes.size // 2 + 5, nodes.size - 1]]:
        acc = np.zeros(p)
        for c in range(4):   # M2M, then the two pseudo-inverse factors
            acc = _chain(blocks[2 + c], mult[row[child[g]] + c], acc)
        for c in range(2):
            acc = _chain(blocks[c], acc, np.zeros(p))
        assert np.array_equal(acc, mult[row[g], :p]), int(g)
        assert not mult[row[g], p:].any()


def _points(right):
    """A point in each depth-8 cell of the left half (leaf capacity 16: leaves
    at depth 6), and right five per depth-8 cell of the right half."""
    rng = np.random.default_rng(4)
    g = np.stack(np.meshgrid(np.arange(128), np.arange(256), indexing="ij"), -1).reshape(-1, 2)
    left = (g + rng.uniform(0.1, 0.9, (g.shape[0], 2))) / 256
    if not right:
        return left
    r = np.repeat(g + np.array([128, 0]), 5, axis=0)
    return np.concatenate([left, (r + rng.uniform(0.1, 0.9, (r.shape[0], 2))) / 256])


@pytest.mark.parametrize("kind,p", [("laplace", 64), ("laplace", 32), ("dipole", 64),
                                    ("helmholtz", 64), ("stokes", 64), ("stokes", 32)])
def test_s2m_of_mixed_plans_does_not_depend_on_the_number_of_leaves(kind, p):
    import torch
    from flexmm_amd import _lib, kernels
    from flexmm_amd.kifmm2d import FMM, StokesFMM, the_help
    the_help.clear()
    rng = np.random.default_rng(5)
    dens = rng.standard_normal((4, _points(True).shape[0]))
    got = []
    for right in (False, True):
        pts = _points(right)
        x, y, n = pts[:, 0].copy(), pts[:, 1].copy(), pts.shape[0]
        q = dens[:, :n]
        print("S2M", kind, p, n, flush=True)
        if kind == "stokes":
            f = StokesFMM(x, y, p, 16, bbox=[0, 1, 0, 1], precision="mixed")
            f.build_expansions(q[0].copy(), q[1].copy())
        else:
            ker = kernels.modified_helmholtz(5.0)[0] if kind == "helmholtz" else kernels.laplace
            f = FMM(x, y, ker, 16, p, bbox=[0, 1, 0, 1], precision="mixed")
            if kind == "dipole":
                f.register_upwardor(kernels.laplace_slp_dlp, "slp+dlp")
                f.build_expansions(q[:2].copy(), "slp+dlp", q[2:].copy())
            else:
                f.build_expansions(q[0].copy())
        t = f.tree
        assert (t.n_s2m > SPLIT_LEAVES) == right

        def tree(name, count, dtype):
            a = torch.empty(count, dtype=dtype, device="cuda")
            _lib.check(f.lib.fmm2d_tree_export(f.handle, _lib.TREE_ARRAYS[name], a.data_ptr(),
                                               a.numel() * a.element_size(), None))
            return a.cpu().numpy()
        a = {k: tree(k, t.n_nodes, torch.int32) for k in ("level", "flags", "bot", "top", "row")}
        code, perm = tree("code", t.n_nodes, torch.int64), tree("perm", n, torch.int32)
        check = torch.empty(t.n_rows * t.PD, dtype=torch.float64, device="cuda")
        _lib.check(f.lib.fmm2d_export_expansions(f.handle, _lib.EXP_ARRAYS["check"],
                                                 check.data_ptr(), check.numel(), None))
        check = check.cpu().numpy().reshape(-1, t.PD)
        leaf = {}
        for g in np.flatnonzero((a["level"] == 6) & (a["flags"] & _lib.NF_UP != 0)):
            leaf[int(code[g])] = (perm[a["bot"][g]:a["top"][g]], check[a["row"][g]])
        got.append(leaf)
        f.close()
    same = [c for c in got[0] if c in got[1] and np.array_equal(got[0][c][0], got[1][c][0])]
    assert len(same) > 1500 and all(got[0][c][0].size == 16 for c in same)
    assert all(np.array_equal(got[0][c][1], got[1][c][1]) for c in same)
