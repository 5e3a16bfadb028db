"""glu_solve recorded into a caller's graph by a plan that has not solved yet:
nothing is allocated in the capture, and every replay gives the same solve."""

import numpy as np
import pytest

from helpers import backward_error, mna_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("name", ["mna600", "small", "grad"])
def test_first_solve_in_a_capture(name, transpose):
    import scipy.sparse as sp
    import torch
    from oracle import oracle as O
    from pyglu import mna
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    data, indices, indptr, n = mna_case(name)
    an = Analysis(data, indices, indptr, n)
    plan, pat = Plan(an), O.SymPattern(an)
    lu = plan.refresh(torch.from_numpy(data).cuda()).reshape(-1)
    plan.factor(lu)
    f = lu.cpu().numpy()
    b = torch.zeros(n, dtype=torch.float32, device="cuda")
    x = torch.zeros_like(b)
    torch.cuda.synchronize()
    print(f"[{name}] n={n} transpose={transpose}", flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan.solve(lu, b, x, transpose=transpose)
    A = sp.csc_matrix((data, indices, indptr), shape=(n, n))
    A = sp.csc_matrix(A.T) if transpose else A
    for seed in (1, 2, 1):
        bh = mna.rhs(n, seed).astype(np.float32)
        b.copy_(torch.from_numpy(bh))
        g.replay()
        got = x.cpu().numpy()
        if not transpose:
            want = O.solve_f32(pat, f, an.col_perm, an.row_perm_inv, an.col_scale_perm, an.row_scale, bh)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        # an eager call (the first of this plan) between the replays
        eager = plan.solve(lu, b, transpose=transpose).cpu().numpy()
        if not transpose:
            assert np.array_equal(got.view(np.uint32), eager.view(np.uint32))
        # single precision factors and solve: n roundings of 2^-24 at most
        for v in (got, eager):
            assert backward_error(A.data, A.indices, A.indptr, n, v.astype(np.float64), bh.astype(np.float64)) <= n * 2.0 ** -24
