"""Batches and groups of orders beyond LDS whose sweeps have many long rows (a
mesh): rows wait for rows of other waves all the time, and every call ends
with every matrix refined."""

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import backward_error

pytestmark = pytest.mark.gpu


def _mesh(m):
    one, line = sp.identity(m), sp.diags([-1.0, 2.0, -1.0], [-1, 0, 1], (m, m))
    A = sp.csc_matrix(sp.kron(one, line) + sp.kron(line, one))
    A.sort_indices()
    return A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32), m * m


@pytest.mark.parametrize("m,count,calls", [(210, 32, 20), (300, 32, 8)])
def test_every_call_refines_every_matrix(m, count, calls):
    import torch
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    data, indices, indptr, n = _mesh(m)
    plan = Plan(Analysis(data, indices, indptr, n))
    rng = np.random.default_rng(m)
    ax = torch.from_numpy(data[None, :] * rng.uniform(0.99, 1.01, (count, data.size))).cuda()
    b = torch.from_numpy(rng.uniform(-1, 1, (count, n))).cuda()
    first = None
    for call in range(calls):
        print(f"n={n} call {call}", flush=True)
        x, _, iters, eta = plan.batch_solve(ax, b, tol=1e-10, maxit=20)
        assert bool((eta <= 1e-10).all()), eta
        if first is None:
            first = x.clone()
            for k in (0, count - 1):
                assert backward_error(ax[k].cpu().numpy(), indices, indptr, n, x[k].cpu().numpy(), b[k].cpu().numpy()) <= 1.1e-10
        assert torch.equal(first.view(torch.int64), x.view(torch.int64))
