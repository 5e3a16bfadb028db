"""Products with A and A' in one workgroup: rows of 1, 7..9, 16/17 and 63..65
entries (eight a pass; beyond 64 a wave's row) and orders around one and two
chunks of 64 rows."""

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import backward_error

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lens", [
    (1, (1,)), (2, (1, 2)), (63, (1, 7, 8, 9)), (64, (16, 17, 1)), (65, (63, 64, 65)),
    (128, (1, 8, 63, 64)), (129, (65, 129, 9)), (1100, (7, 8, 9, 15, 16, 17, 63, 64, 65, 500, 1))])
@pytest.mark.parametrize("transpose", [False, True])
def test_residual_of_row_lengths(n, lens, transpose):
    """One preconditioner solve leaves an FP32-sized residual; the backward
    error the device takes from its own products equals the host's.  Each side
    rounds a row of k entries by at most (k + 4) 2^-53 (|A| |x| + |b|), and both
    divide by |A| |x| + |b|: they agree within 4 (k + 8) 2^-53."""
    import torch
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    rng = np.random.default_rng(n + len(lens))
    A = sp.lil_matrix((n, n))
    for i in range(n):
        ln = min(lens[i % len(lens)] if i < 4 * len(lens) else 1 + i % 4, n)
        cols = rng.choice(n, size=ln, replace=False)
        A[i, cols] = rng.uniform(-1, 1, ln) / ln
        A[i, i] = 3.0 + rng.uniform(0, 1)
    A = sp.csc_matrix(sp.csc_matrix(A).T if transpose else A)
    A.sort_indices()
    data, indices, indptr = A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32)
    plan = Plan(Analysis(data, indices, indptr, n))
    ax = torch.from_numpy(data).cuda()
    lu = plan.refresh(ax).reshape(-1).clone()
    plan.factor(lu)
    b = rng.uniform(-1, 1, n)
    x, it, eta = plan.refine(ax, lu, torch.from_numpy(b).cuda(), tol=0.0, maxit=1, transpose=transpose)
    M = sp.csc_matrix(A.T) if transpose else A
    host = backward_error(M.data, M.indices, M.indptr, n, x.cpu().numpy(), b)
    k = int(np.diff(sp.csr_matrix(M).indptr).max())
    print(f"n={n} transpose={transpose} longest row {k}: eta {eta:.17e} host {host:.17e}", flush=True)
    assert it == 1
    assert abs(eta - host) <= 4 * (k + 8) * 2.0 ** -53
