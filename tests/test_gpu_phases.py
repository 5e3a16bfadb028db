"""Phases of the factorization (leading steps in independent components, a
workgroup each, later entries' products subtracted afterwards) on patterns
whose windows leave most steps to them: products of 1, 32, 33 and many columns
an entry, unsymmetric patterns, columns without L entries."""

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import mna_case

pytestmark = pytest.mark.gpu


def _blocks(sizes, rails, seed):
    """Independent tridiagonal blocks, each joined to the same rails: every
    rail entry gets a product from every block's columns."""
    rng = np.random.default_rng(seed)
    n = sum(sizes) + rails
    A = sp.lil_matrix((n, n))
    at = 0
    for s in sizes:
        for i in range(s):
            A[at + i, at + i] = rng.uniform(2, 4)
            if i:
                A[at + i, at + i - 1] = rng.uniform(-1, 1)
                A[at + i - 1, at + i] = rng.uniform(-1, 1)
        for r in range(n - rails, n):
            A[r, at + s - 1] = rng.uniform(-1, 1)
            A[at + s - 1, r] = rng.uniform(-1, 1)
        at += s
    for r in range(n - rails, n):
        for c in range(n - rails, n):
            A[r, c] = rng.uniform(-1, 1) + (3.0 * len(sizes) if r == c else 0)
    A = sp.csc_matrix(A)
    A.sort_indices()
    return A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32), n


def _unsym(n, seed):
    """Unsymmetric, with a dense row, a dense column and columns that end up
    without L entries."""
    rng = np.random.default_rng(seed)
    A = sp.random(n, n, density=2.5 / n, random_state=seed, format="lil")
    for i in range(n):
        A[i, i] = 3.0 + rng.uniform(0, 1)
    for c in rng.choice(n, 40, replace=False):
        A[n // 2, c] = rng.uniform(-0.1, 0.1)
    for r in rng.choice(n, 40, replace=False):
        A[r, n // 3] = rng.uniform(-0.1, 0.1)
    A = sp.csc_matrix(A)
    A.sort_indices()
    return A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32), n


CASES = {
    "one": lambda: _blocks([6], 8, 1), "few": lambda: _blocks([5, 6, 7, 8], 9, 2),
    "lane": lambda: _blocks([8] * 32, 10, 3), "wave": lambda: _blocks([8] * 33, 10, 4),
    "many": lambda: _blocks([3, 9, 17] * 100, 12, 5), "unsym300": lambda: _unsym(300, 6),
    "unsym1500": lambda: _unsym(1500, 7), "mna2k": lambda: mna_case("mna2k"), "add32": lambda: mna_case("add32"),
    "grad": lambda: mna_case("grad"),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("values", [60, 700])
def test_phases_match_oracle(name, values):
    """One LDS window of few values at the end: the steps before it run as
    phases.  Factors equal the oracle's bit for bit with and without GESP, on
    two value sets of one plan."""
    import torch
    from oracle import oracle as O
    from pyglu import mna
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    data, indices, indptr, n = CASES[name]()
    an = Analysis(data, indices, indptr, n)
    plan, pat = Plan(an, lds_windows=1, lds_window_values=values), O.SymPattern(an)
    print(f"[{name}] n={n} levels={an.num_lev} segments={plan.segments} windows={plan.lds_window_count} "
          f"(steps {plan.lds_window_steps})", flush=True)
    factor = O.factor_f32_sparse if hasattr(O, "factor_f32_sparse") and n > 10000 else O.factor_f32
    for seed, perturb in ((1, False), (2, True)):
        lu = plan.refresh(torch.from_numpy(mna.perturb_values(data, seed)).cuda()).reshape(-1)
        want = factor(pat, lu.cpu().numpy(), perturb=perturb)[0]
        plan.factor(lu, perturb=perturb)
        assert np.array_equal(lu.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("perturb", [False, True])
@pytest.mark.parametrize("split", [0, 1])
def test_group_phases_match_single_path(split, perturb):
    """Members with and without phases in one group: every member's factors
    equal its own single-path factors, twice on other value sets, and every
    backward error meets the tolerance."""
    import torch
    from pyglu import mna
    from pyglu.analysis import Analysis
    from pyglu.device import Group, Plan
    mats = [CASES[k]() for k in ("unsym1500", "many", "mna2k", "lane", "one")] + [mna_case("small")]
    plans = [Plan(Analysis(*m), lds_windows=1, lds_window_values=700) for m in mats]
    plans.append(Plan(Analysis(*mats[2])))   # one window, no phase
    mats.append(mats[2])
    g = Group(plans, split=split)
    for seed in (1, 2):
        axs = [torch.from_numpy(mna.perturb_values(m[0], seed)).cuda() for m in mats]
        bs = [torch.from_numpy(mna.rhs(m[3], seed)).cuda() for m in mats]
        xs, lus, iters, eta = g.solve(axs, bs, tol=1e-10, maxit=20, perturb=perturb)
        for i, (p, ax) in enumerate(zip(plans, axs)):
            lu = p.refresh(ax).reshape(-1)
            p.factor(lu, perturb=perturb)
            assert torch.equal(lu.view(torch.int32), lus[i].view(torch.int32)), (seed, i)
        assert float(eta.max()) <= 1e-10
    g.close()
