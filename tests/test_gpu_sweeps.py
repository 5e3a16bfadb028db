"""Triangular sweeps with the vector in LDS at the sizes where their tasks
change shape: rows of 6/7, 16/17, 32/33 and 64/65 entries (a lane each, then
16, 32 and 64 lanes a row, then several passes), orders around one wave, and
values that could be taken for a row that is not done."""

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import backward_error

pytestmark = pytest.mark.gpu


def _case(n, lens, seed):
    """A tridiagonal matrix of order n whose last rows and columns have the
    given numbers of off-diagonal entries."""
    rng = np.random.default_rng(seed)
    A = sp.lil_matrix((n, n))
    for i in range(n):
        A[i, i] = 4.0 + rng.uniform(0, 1)
        if i:
            A[i, i - 1] = rng.uniform(-1, 1)
            A[i - 1, i] = rng.uniform(-1, 1)
    for k, ln in enumerate(lens):
        r = n - 1 - k
        if r <= 0:
            break
        for c in rng.choice(r, size=min(ln, r), replace=False):
            A[r, c] = rng.uniform(-0.1, 0.1)
            A[c, r] = rng.uniform(-0.1, 0.1)
        A[r, r] = 4.0 + 0.1 * ln
    A = sp.csc_matrix(A)
    A.sort_indices()
    return A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32), n


@pytest.mark.parametrize("n,lens", [
    (1, ()), (2, ()), (63, (6, 7)), (64, (15, 16, 17)), (65, (31, 32, 33)), (130, (63, 64, 65)),
    (700, (6, 7, 16, 17, 32, 33, 64, 65, 127, 128, 129, 320, 321, 385)), (2049, (1000, 1500, 449, 511, 513))])
def test_sweeps_at_task_edges(n, lens):
    """The exact solve equals the oracle bit for bit; the refinement of A and
    A' converges to a host-checked backward error."""
    import torch
    from oracle import oracle as O
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    data, indices, indptr, n = _case(n, lens, 77 + n)
    an = Analysis(data, indices, indptr, n)
    plan, pat = Plan(an), O.SymPattern(an)
    lu = torch.from_numpy(an.val.copy()).cuda()
    plan.factor(lu)
    b = np.random.default_rng(n).uniform(-1, 1, n)
    b32 = b.astype(np.float32)
    x = plan.solve(lu, torch.from_numpy(b32).cuda()).cpu().numpy()
    want = O.solve_f32(pat, lu.cpu().numpy(), an.col_perm, an.row_perm_inv, an.col_scale_perm, an.row_scale, b32)
    assert np.array_equal(x.view(np.uint32), want.view(np.uint32))
    ax = torch.from_numpy(data).cuda()
    for transpose in (False, True):
        xr, it, eta = plan.refine(ax, lu, torch.from_numpy(b).cuda(), tol=1e-12, maxit=20, transpose=transpose)
        A = sp.csc_matrix((data, indices, indptr), shape=(n, n))
        At = sp.csc_matrix(A.T) if transpose else A
        eta_h = backward_error(At.data, At.indices, At.indptr, n, xr.cpu().numpy(), b)
        print(f"n={n} transpose={transpose} solves={it} eta={eta:.1e} host {eta_h:.1e}", flush=True)
        assert eta <= 1e-12 and eta_h <= 2e-12


@pytest.mark.parametrize("bits", [0x7f8a5ca1, 0x7fca5ca1, 0xffffffff, 0x7f800000])
def test_sweeps_with_non_finite_values(bits):
    """NaN (also the pattern that marks a row as not done) and infinite
    factors and right-hand sides: every row completes, with the oracle's
    finite and non-finite entries."""
    import torch
    from oracle import oracle as O
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    n = 300
    data, indices, indptr, n = _case(n, (7, 20, 40, 70, 200), 5)
    an = Analysis(data, indices, indptr, n)
    plan, pat = Plan(an), O.SymPattern(an)
    lu = torch.from_numpy(an.val.copy()).cuda()
    plan.factor(lu)
    good = lu.cpu().numpy()
    bad = np.array([bits], np.uint32).view(np.float32)[0]
    for where in ("rhs", "factor"):
        b = np.random.default_rng(1).uniform(-1, 1, n).astype(np.float32)
        f = good.copy()
        if where == "rhs":
            b[n // 2] = bad
        else:
            f[an.l_col_ptr[n // 2]] = bad   # a pivot
        x = plan.solve(torch.from_numpy(f).cuda(), torch.from_numpy(b).cuda()).cpu().numpy()
        with np.errstate(all="ignore"):
            want = O.solve_f32(pat, f, an.col_perm, an.row_perm_inv, an.col_scale_perm, an.row_scale, b)
        fin = np.isfinite(want)
        assert np.array_equal(fin, np.isfinite(x)) and np.array_equal(np.isnan(x), np.isnan(want))
        assert np.array_equal(x[fin].view(np.uint32), want[fin].view(np.uint32))


def _solve_transposed(an, lu, b):
    """A' x = b with the FP32 factors, row by row in order: U' forward with
    the pivot division, then L' backward."""
    one = np.float32
    t = (b[an.row_perm].astype(np.float64) * an.row_scale[an.row_perm]).astype(one)
    cp, ri, ld = an.sym_c_ptr.tolist(), an.sym_r_idx.tolist(), an.l_col_ptr.tolist()
    for r in range(an.n):
        acc = t[r]
        for q in range(cp[r], ld[r]):
            acc = acc - lu[q] * t[ri[q]]
        t[r] = acc / lu[ld[r]]
    for r in range(an.n - 1, -1, -1):
        acc = t[r]
        for q in range(cp[r + 1] - 1, ld[r], -1):
            acc = acc - lu[q] * t[ri[q]]
        t[r] = acc
    back = an.col_perm_inv
    return (t[back].astype(np.float64) * an.col_scale_perm[back]).astype(one)


@pytest.mark.parametrize("name", ["mna600", "small", "batch", "grad"])
def test_solves_are_sequential(name):
    """A x = b and A' x = b (n=50k "grad": split over many workgroups) equal
    the row-by-row solve bit for bit, with a second value set and right-hand
    side over the same plan; the refinement of A' reaches its tolerance."""
    import torch
    from helpers import mna_case
    from oracle import oracle as O
    from pyglu import mna
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    data, indices, indptr, n = mna_case(name)
    an = Analysis(data, indices, indptr, n)
    plan, pat = Plan(an), O.SymPattern(an)
    for seed in (1, 2):
        ax = torch.from_numpy(mna.perturb_values(data, seed)).cuda()
        lu = plan.refresh(ax).reshape(-1)
        plan.factor(lu)
        b = mna.rhs(n, seed).astype(np.float32)
        f = lu.cpu().numpy()
        x = plan.solve(lu, torch.from_numpy(b).cuda()).cpu().numpy()
        want = O.solve_f32(pat, f, an.col_perm, an.row_perm_inv, an.col_scale_perm, an.row_scale, b)
        assert np.array_equal(x.view(np.uint32), want.view(np.uint32))
        xt = plan.solve(lu, torch.from_numpy(b).cuda(), transpose=True).cpu().numpy()
        assert np.array_equal(xt.view(np.uint32), _solve_transposed(an, f, b).view(np.uint32))
    x, it, eta = plan.refine(ax, lu, torch.from_numpy(b.astype(np.float64)).cuda(), tol=1e-11, maxit=20, transpose=True)
    print(f"[{name}] n={n} transposed refinement {it} solves eta {eta:.1e}", flush=True)
    assert eta <= 1e-11
