"""The sweeps' division (reciprocal taken ahead, the full division for operands
outside [2^-30, 2^30) and [2^-64, 2^64)) at the edges of those ranges, among
the smallest and largest values and below the normal range: the exact solves
equal the oracle's quotients bit for bit."""

import numpy as np
import pytest

from helpers import mna_case
from test_gpu_sweeps import _solve_transposed

pytestmark = pytest.mark.gpu


def _around(rng, exps, count):
    """`count` values at the given powers of two: exactly, one unit in the
    last place to either side, or anywhere in the two binades next to them."""
    e = rng.choice(exps, count)
    v = np.ldexp(1.0, e).astype(np.float32)
    kind = rng.integers(0, 4, count)
    v = np.where(kind == 1, np.nextafter(v, np.float32(0)), v)
    v = np.where(kind == 2, np.nextafter(v, np.float32(np.inf)), v)
    v = np.where(kind == 3, (v * rng.uniform(0.5, 2, count)).astype(np.float32), v)
    return (v * rng.choice(np.float32([1, -1]), count)).astype(np.float32)


def _finite(v):
    v = v.astype(np.float32)
    return np.where(np.isfinite(v), v, np.float32(1))


PIVOTS = {"edges": [-31, -30, -29, 29, 30, 31], "extremes": [-149, -140, -127, -126, -125, 100, 126, 127],
          "middle": [-2, -1, 0, 1, 2]}
VALUES = {"edges": [-65, -64, -63, 63, 64, 65], "extremes": [-149, -140, -127, -126, -125, 120, 126, 127],
          "middle": [-2, 0, 2]}


@pytest.mark.parametrize("name", ["mna2k", "grad"])
@pytest.mark.parametrize("pivots", list(PIVOTS))
@pytest.mark.parametrize("values", list(VALUES))
def test_quotients(name, pivots, values):
    """Factors of a diagonal (every other entry 0): a row's value is its
    right-hand side's quotient by its pivot."""
    import torch
    from oracle import oracle as O
    from pyglu.analysis import Analysis
    from pyglu.device import Plan
    data, indices, indptr, n = mna_case(name)
    an = Analysis(data, indices, indptr, n)
    plan, pat = Plan(an), O.SymPattern(an)
    rng = np.random.default_rng(len(pivots) * 16 + len(values))
    for seed in range(2):
        f = np.zeros(an.nnz_lu, np.float32)
        d = _around(rng, PIVOTS[pivots], n)
        f[an.l_col_ptr] = d = np.where(d == 0, np.float32(2.0 ** -149), d)
        row = _around(rng, VALUES[values], n)
        with np.errstate(all="ignore"):   # quotients that overflow would make NaN of every row after them
            row = np.where(np.isfinite(row / d) & (np.abs(row / d) < 2.0 ** 90), row, d * rng.uniform(0.5, 2, n).astype(np.float32))
            row = row.astype(np.float32)
        lu = torch.from_numpy(f).cuda()
        with np.errstate(all="ignore"):
            # right-hand sides whose scaled values are about `row`, row by row
            b = np.zeros(n, np.float32)
            b[an.col_perm] = _finite(row / an.col_scale_perm)
            want = O.solve_f32(pat, f, an.col_perm, an.row_perm_inv, an.col_scale_perm, an.row_scale, b)
        got = plan.solve(lu, torch.from_numpy(b).cuda()).cpu().numpy()
        nan = np.isnan(want)
        assert np.array_equal(nan, np.isnan(got))
        assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
        if name == "mna2k":
            with np.errstate(all="ignore"):
                b[an.row_perm] = _finite(row / an.row_scale[an.row_perm])
                want = _solve_transposed(an, f, b)
            got = plan.solve(lu, torch.from_numpy(b).cuda(), transpose=True).cpu().numpy()
            nan = np.isnan(want)
            assert np.array_equal(nan, np.isnan(got))
            assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
    print(f"[{name}] pivots {pivots} values {values}: {int(nan.sum())} of {n} NaN, "
          f"{int(np.isinf(want).sum())} infinite, {int((want == 0).sum())} zero", flush=True)
