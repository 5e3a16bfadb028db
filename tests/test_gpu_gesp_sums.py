"""GESP column sums (src/numeric.cu:490-506) of columns around the lengths where
a column changes hands: 64 entries (a lane, then a wave) and the 64- and
256-entry passes of a wave.  A replaced pivot carries the value into the
factors, which are compared with the oracle bit for bit."""

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [1, 63, 64, 65, 128, 129, 256, 257, 321, 512, 600, 1500])
def test_gesp_value_of_long_columns(length):
    """An arrow matrix whose last column has `length` entries and holds the
    largest sum; one pivot is drifted to almost zero.  Single path, workgroup
    batch and interleaved batch (more than 1,024 columns in the first step)."""
    import torch
    from oracle import oracle as O
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    rng = np.random.default_rng(length)
    n = 1500
    A = sp.lil_matrix((n, n))
    for i in range(n):
        A[i, i] = rng.uniform(1, 2)
        if i < n - 1:
            A[n - 1, i] = rng.uniform(0.1, 1)
        if i >= n - length:
            A[i, n - 1] = rng.uniform(0.5, 1)
    A[n - 1, n - 1] = 3.0 * n
    A = sp.csc_matrix(A)
    A.sort_indices()
    data, indices, indptr = A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32)
    an = Analysis(data, indices, indptr, n)
    pat = O.SymPattern(an)
    drift = data * (1 + rng.uniform(-0.1, 0.1, data.size))
    for c in (3, n // 2):
        drift[indptr[c] + np.flatnonzero(indices[indptr[c]:indptr[c + 1]] == c)[0]] = 1e-12
    ax = torch.from_numpy(drift).cuda()
    for windows in (0, -1):
        plan = Plan(an, lds_windows=windows)
        base = plan.refresh(ax).reshape(-1)
        want, pert = O.factor_f32(pat, base.cpu().numpy(), perturb=True)
        assert np.any(want == np.float32(pert))
        lu = base.clone()
        plan.factor(lu, perturb=True)
        assert np.array_equal(lu.cpu().numpy().view(np.uint32), want.view(np.uint32))
        bl = plan.batch_factor(torch.stack([ax] * 3), perturb=True).cpu().numpy()
        print(f"length={length} windows={windows} grid steps={plan.batch_grid_levels} pert={pert:.3e}", flush=True)
        assert all(np.array_equal(row.view(np.uint32), want.view(np.uint32)) for row in bl)
