"""One plan as several members of a group (a block instanced more than once,
with other values): every member works in scratch of its own, whatever runs
beside the fused launch."""

import numpy as np
import pytest

from helpers import backward_error
from test_gpu_phases import CASES

pytestmark = pytest.mark.gpu


def _solve(plans, mats, axs, bs, split, perturb):
    from pyglu.device import Group
    g = Group(plans, split=split)
    out = g.solve(axs, bs, tol=1e-10, maxit=20, perturb=perturb)
    again = g.solve(axs, bs, tol=1e-10, maxit=20, perturb=perturb)
    for a, b in zip(out[0] + out[1], again[0] + again[1]):
        assert np.array_equal(a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32))
    g.close()
    return out


@pytest.mark.parametrize("perturb", [False, True])
@pytest.mark.parametrize("times", [2, 3])
def test_repeated_plan(times, perturb):
    """A plan with phases two and three times, with another one: every
    member's factors equal its own single-path factors bit for bit, and its
    solution is the same bits whatever the split."""
    import torch
    from pyglu import mna
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    big, small = CASES["mna2k"](), CASES["many"]()
    p = Plan(Analysis(*big), lds_windows=1, lds_window_values=700)
    q = Plan(Analysis(*small), lds_windows=1, lds_window_values=700)
    plans, mats = [p] * times + [q, q], [big] * times + [small, small]
    axs = [torch.from_numpy(mna.perturb_values(m[0], 5 + i)).cuda() for i, m in enumerate(mats)]
    bs = [torch.from_numpy(mna.rhs(m[3], 5 + i)).cuda() for i, m in enumerate(mats)]
    want = []
    for r, ax in zip(plans, axs):
        lu = r.refresh(ax).reshape(-1)
        want.append(r.factor(lu, perturb=perturb).view(torch.int32))
    first = None
    for split in (0, 1, 2):
        print(f"times={times} perturb={perturb} split={split}", flush=True)
        xs, lus, iters, eta = _solve(plans, mats, axs, bs, split, perturb)
        for w, lu in zip(want, lus):
            assert torch.equal(w, lu.view(torch.int32))
        assert float(eta.max()) <= 1e-10
        for (data, indices, indptr, n), ax, b, x in zip(mats, axs, bs, xs):
            assert backward_error(ax.cpu().numpy(), indices, indptr, n, x.cpu().numpy(), b.cpu().numpy()) <= 1.1e-10
        if first is None:
            first = [x.clone() for x in xs]
        assert all(torch.equal(a.view(torch.int64), x.view(torch.int64)) for a, x in zip(first, xs))


def test_group_beside_the_plan_on_another_stream():
    """A group on one stream while one of its plans factors on another: both
    give the bits they give alone."""
    import torch
    from pyglu import mna
    from pyglu.analysis import Analysis
    from pyglu.device import Group, Plan
    m = CASES["mna2k"]()
    p = Plan(Analysis(*m), lds_windows=1, lds_window_values=700)
    axs = [torch.from_numpy(mna.perturb_values(m[0], 31 + i)).cuda() for i in range(3)]
    bs = [torch.from_numpy(mna.rhs(m[3], 31 + i)).cuda() for i in range(2)]
    want = [p.factor(p.refresh(ax).reshape(-1)).clone() for ax in axs]
    g = Group([p, p], split=0)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(other):
        lus = [p.refresh(axs[2]).reshape(-1) for _ in range(20)]
        for lu in lus:
            p.factor(lu)
    _, glus, _, eta = g.solve(axs[:2], bs, tol=1e-10, maxit=20)
    torch.cuda.synchronize()
    assert all(torch.equal(lu.view(torch.int32), want[2].view(torch.int32)) for lu in lus)
    assert all(torch.equal(a.view(torch.int32), b.view(torch.int32)) for a, b in zip(glus, want))
    assert float(eta.max()) <= 1e-10
    g.close()
