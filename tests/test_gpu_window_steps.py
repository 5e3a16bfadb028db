"""Steps of an LDS window at the sizes where their chunks change: entries that
2..4 columns of a step update (a lane each), 5..16, 17..32 and more (16 lanes
each, one or several chunks), columns with 1..4 and more updates a lane, and
workgroups of one wave up to sixteen."""

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _bundle(m, rails, seed):
    """m independent columns that all reach the same `rails` rows (so one step
    updates rails x rails entries with m sources each), then a dense block of
    the rails; values spread over four decades."""
    rng = np.random.default_rng(seed)
    n = m + rails
    A = sp.lil_matrix((n, n))
    for i in range(m):
        A[i, i] = 10.0 ** rng.uniform(0, 2)
        for r in range(m, n):
            A[i, r] = 10.0 ** rng.uniform(-2, 0) * rng.choice([-1, 1])
            A[r, i] = 10.0 ** rng.uniform(-2, 0) * rng.choice([-1, 1])
    for r in range(m, n):
        for c in range(m, n):
            A[r, c] = rng.uniform(-1, 1) + (4.0 * n if r == c else 0.0)
    A = sp.csc_matrix(A)
    A.sort_indices()
    return A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32), n


@pytest.mark.parametrize("m,rails", [(1, 1), (2, 5), (3, 6), (4, 5), (5, 7), (16, 6), (17, 5), (32, 6), (33, 5), (64, 9),
                                     (65, 6), (200, 12)])
@pytest.mark.parametrize("threads", [64, 192, 1024])
def test_window_steps_match_oracle(m, rails, threads):
    """Factors bit-identical to the oracle with and without GESP, on the
    single and the batched path, every step in one window."""
    import torch
    from oracle import oracle as O
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    data, indices, indptr, n = _bundle(m, rails, 100 * m + rails)
    an = Analysis(data, indices, indptr, n)
    plan, pat = Plan(an, block_threads=threads), O.SymPattern(an)
    print(f"m={m} rails={rails} levels={an.num_lev} windows={plan.lds_window_count} steps={plan.lds_window_steps}",
          flush=True)
    assert plan.lds_window_count == (rails >= 5)
    ax = torch.from_numpy(data).cuda()
    base = plan.refresh(ax).reshape(-1)
    for perturb in (False, True):
        lu = base.clone()
        plan.factor(lu, perturb=perturb)
        want, _ = O.factor_f32(pat, base.cpu().numpy(), perturb=perturb)
        assert np.array_equal(lu.cpu().numpy().view(np.uint32), want.view(np.uint32))
        bl = plan.batch_factor(torch.stack([ax, ax, ax]), perturb=perturb).cpu().numpy()
        assert all(np.array_equal(row.view(np.uint32), want.view(np.uint32)) for row in bl)
