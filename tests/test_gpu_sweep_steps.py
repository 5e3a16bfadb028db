"""Triangular sweeps a level a step, with more rows of several chunks (257 and
more entries) than a workgroup's waves can have open, and rows whose entries
are set one, two and five steps before their own."""

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import backward_error
from test_gpu_sweeps import _case

pytestmark = pytest.mark.gpu


def _band(n, width):
    """Every row takes the `width` rows before it, so a row's entries are set
    1 .. width steps before its own."""
    rng = np.random.default_rng(n + width)
    A = sp.diags([rng.uniform(-0.5, 0.5, n - abs(k)) / width if k else rng.uniform(4, 5, n)
                  for k in range(-width, width + 1)], list(range(-width, width + 1)), format="csc")
    A.sort_indices()
    return A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32), n


@pytest.mark.parametrize("make", [
    lambda: _case(1300, tuple(range(257, 557, 10)), 11), lambda: _case(700, (256, 257, 512, 513) * 4, 12),
    lambda: _case(400, (300,), 13), lambda: _band(120, 1), lambda: _band(150, 4), lambda: _band(150, 5),
    lambda: _band(200, 17), lambda: _band(300, 63), lambda: _band(300, 70)])
def test_sweeps_by_steps(make):
    """The exact solve equals the oracle bit for bit; the refinement of A and
    A' converges to a host-checked backward error."""
    import torch
    from oracle import oracle as O
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    data, indices, indptr, n = make()
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
