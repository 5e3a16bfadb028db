"""Divisions and value copies of a group's members, spread over many workgroups
a member: none (a diagonal), a few, and more items than one pass of all the
workgroups takes, with and without replaced pivots."""

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _member(n, tail, seed):
    """A diagonal with `tail` dense last rows and columns."""
    rng = np.random.default_rng(seed)
    A = sp.lil_matrix((n, n))
    A.setdiag(rng.uniform(2, 3, n))
    for i in range(n - tail, n):
        A[i, :i] = rng.uniform(0.1, 1, i) / n
        A[:i, i] = rng.uniform(0.1, 1, i)[:, None] / n
        A[i, i] = 4.0
    A = sp.csc_matrix(A)
    A.sort_indices()
    return A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32), n


@pytest.mark.parametrize("perturb", [False, True])
@pytest.mark.parametrize("split", [0, 1])
def test_group_factors_equal_single_path(split, perturb):
    """Every member's factors equal its own single-path factors bit for bit,
    and, without replaced pivots, every backward error meets the tolerance."""
    import torch
    from pyglu.analysis import Analysis
    from pyglu.device import Group, Plan
    mats = [_member(1, 0, 1), _member(100, 0, 2), _member(63, 1, 3), _member(257, 3, 4), _member(1500, 12, 5)]
    plans = [Plan(Analysis(*m)) for m in mats]
    g = Group(plans, split=split)
    axs = []
    for data, indices, indptr, n in mats:
        v = data.copy()
        if perturb and n > 1:   # a pivot to be replaced
            v[indptr[n // 2] + np.flatnonzero(indices[indptr[n // 2]:indptr[n // 2 + 1]] == n // 2)[0]] = 1e-12
        axs.append(torch.from_numpy(v).cuda())
    bs = [torch.from_numpy(np.random.default_rng(m[3]).uniform(-1, 1, m[3])).cuda() for m in mats]
    xs, lus, iters, eta = g.solve(axs, bs, tol=1e-10, maxit=20, perturb=perturb)
    for i, (p, ax) in enumerate(zip(plans, axs)):
        lu = p.refresh(ax).reshape(-1)
        p.factor(lu, perturb=perturb)
        print(f"n={mats[i][3]} split={split} perturb={perturb} eta={float(eta[i]):.1e}", flush=True)
        assert torch.equal(lu.view(torch.int32), lus[i].view(torch.int32))
    if not perturb:
        assert float(eta.max()) <= 1e-10
    g.close()
