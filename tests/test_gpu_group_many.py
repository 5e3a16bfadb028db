"""Groups of about as many members as a launch may have blocks in its second
dimension (65,536), and more."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [65_535, 65_536, 66_000])
def test_many_members(count):
    """Members of order 3, all of one plan, each with its own values."""
    import torch
    from pyglu.analysis import Analysis
    from pyglu.device import Group, Plan
    A = np.array([[4.0, 1.0, 0.0], [1.0, 5.0, 2.0], [0.0, 2.0, 6.0]])
    indptr, indices = np.array([0, 2, 5, 7], np.int32), np.array([0, 1, 0, 1, 2, 1, 2], np.int32)
    data = np.array([4.0, 1.0, 1.0, 5.0, 2.0, 2.0, 6.0])
    plan = Plan(Analysis(data, indices, indptr, 3))
    g = Group([plan] * count, split=0)
    scale = 1.0 + np.arange(count) / count
    ax = torch.from_numpy(scale[:, None] * data[None, :]).cuda()
    b = torch.from_numpy(np.tile([1.0, 2.0, 3.0], (count, 1))).cuda()
    print(f"{count} members", flush=True)
    xs, _, _, eta = g.solve(list(ax), list(b), tol=1e-12, maxit=10)
    x = torch.stack(xs).cpu().numpy()
    want = np.linalg.solve(A, [1.0, 2.0, 3.0])[None, :] / scale[:, None]
    assert float(eta.max()) <= 1e-12
    # backward error 1e-12 with a condition number below 10
    assert np.abs(x - want).max() <= 1e-10
    g.close()
