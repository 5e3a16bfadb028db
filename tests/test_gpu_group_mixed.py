"""Members in LDS behind an odd order beyond it in one group: their value
copies start on whole lines whatever the copies before them take."""

import numpy as np
import pytest

from helpers import backward_error, mna_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("odd", [39991, 39993, 39995])
def test_small_members_behind_an_odd_order(odd):
    """The small members' factors and solutions are the same bits with and
    without the large member before them."""
    import torch
    from pyglu import mna
    from pyglu.analysis import Analysis
    from pyglu.device import Group, Plan
    large = mna.mna_csc(mna.MNASpec(n_nodes=odd - 40, n_vsrc=40, n_rails=3, rail_deg=120), 7)
    mats = [large, mna_case("mna600"), mna_case("mna2k")]
    assert large[3] == odd
    plans = [Plan(Analysis(*m)) for m in mats]
    axs = [torch.from_numpy(mna.perturb_values(m[0], 3)).cuda() for m in mats]
    bs = [torch.from_numpy(mna.rhs(m[3], 3)).cuda() for m in mats]
    print(f"n={odd}", flush=True)
    out = []
    for k in (0, 1):
        g = Group(plans[k:], split=0)
        xs, lus, _, eta = g.solve(axs[k:], bs[k:], tol=1e-10, maxit=20)
        assert float(eta.max()) <= 1e-10
        out.append((xs[1 - k:], lus[1 - k:]))
        if k == 0:
            data, indices, indptr, n = large
            assert backward_error(axs[0].cpu().numpy(), indices, indptr, n, xs[0].cpu().numpy(), bs[0].cpu().numpy()) <= 1.1e-10
        g.close()
    for a, b in zip(out[0][0] + out[0][1], out[1][0] + out[1][1]):
        assert np.array_equal(a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32))
