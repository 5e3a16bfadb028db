"""Workloads of the library's public entry points, for timing.

A case is one pass of a circuit simulator's inner loop on modified-nodal-
analysis (MNA) matrices of ``pyglu.mna``: the pattern is analysed and planned
once (``prepare``), then every pass (``run``) brings new values and goes
through the device API:

``newton``    refresh + FP32 factor + FP32 solve (the drop-in path), one matrix
``resolve``   FP32 solve with kept factors, A x = b or A' x = b, one matrix
``refined``   refresh + factor + FP64-refined solve, one matrix
``autograd``  forward + backward of the differentiable solve
``batch``     many value sets of one pattern: refresh + factor + refined solve
``refactor``  many value sets of one pattern: refresh + factor only
``group``     distinct patterns in one launch: refresh + factor + refined solve

Value sets drift by up to 10% around the analysed ones, as a Newton step's
do; right-hand sides are uniform in [-1, 1].
"""

from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "glu-hcu_amd"))

from pyglu import mna                                    # noqa: E402
from pyglu.analysis import Analysis, analyze_many        # noqa: E402
from pyglu.device import Group, Plan, spsolve_autograd   # noqa: E402


# --------------------------------------------------------------------------
# cases
# --------------------------------------------------------------------------

def _case(name, kind, n, extra, rails, rail_deg, pattern, count=1, perturb=False, graph=False, transpose=False,
          tol=1e-10):
    c = {"kind": kind, "n": n, "extra": extra, "rails": rails, "rail_deg": rail_deg, "pattern": pattern,
         "count": count, "perturb": perturb, "graph": graph, "transpose": transpose, "tol": tol}
    return {"name": name, **c} if name else c


def listed():
    return [
        # a small subcircuit: the smallest call, launches and latency only
        _case("newton-640", "newton", 640, 3, 2, 40, 1),
        # the order of the reference's example input, replayed from graphs
        # (a fixed program that steps in place)
        _case("newton-4960-graph", "newton", 4960, 3, 3, 300, 1, graph=True),
        # a mid-sized circuit with GESP, as a user without a good pivot order
        # runs it
        _case("newton-20000-gesp", "newton", 20000, 5, 5, 1000, 3, perturb=True),
        # the largest single factorization and solve: an extracted netlist
        _case("newton-200003", "newton", 200003, 7, 20, 2000, 2),
        # factors kept over many right-hand sides, vector beyond LDS
        _case("resolve-50000", "resolve", 50000, 5, 10, 2000, 5),
        # adjoint sensitivities with kept FP32 factors
        _case("resolve-4960-adjoint", "resolve", 4960, 3, 3, 300, 1, transpose=True),
        # an accurate solve of one large system
        _case("refined-100000", "refined", 100000, 7, 10, 1000, 2),
        # an accurate solve to near FP64, odd order
        _case("refined-9973-tight", "refined", 9973, 4, 3, 250, 17, tol=1e-13),
        # training through the solve
        _case("autograd-50000", "autograd", 50000, 5, 10, 2000, 5, tol=1e-13),
        # Monte-Carlo / corner runs of one circuit, the chip full
        _case("batch-256x20000", "batch", 20000, 5, 5, 1000, 3, count=256),
        # a partial group of corners of a small circuit, values only
        _case("refactor-37x3001-gesp", "refactor", 3001, 3, 3, 75, 11, count=37, perturb=True),
        # a netlist partitioned into distinct blocks
        _case("group-16", "group", 30000, 4, 3, 0, 4000, count=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["newton", "newton", "resolve", "refined", "autograd", "batch", "refactor", "group"])
    top = {"newton": 150000, "resolve": 150000, "refined": 80000, "autograd": 45000, "batch": 19000,
           "refactor": 19000, "group": 28000}[kind]
    n = _log(rng, 600, top)
    rails = rng.randint(2, 5) if n < 30000 else rng.randint(5, 12)
    extra = rng.randint(3, 5)
    count = 1
    if kind in ("batch", "refactor"):
        count = _log(rng, 1, 250)
    elif kind == "group":
        count = rng.randint(2, 14)
    return _case("", kind, n, extra, rails, max(8, n // rng.randint(20, 100)) if kind != "group" else 0,
                 rng.randint(1, 10 ** 6), count=count,
                 perturb=kind not in ("resolve", "refined", "autograd") and rng.random() < 0.3,
                 graph=kind in ("newton", "resolve") and rng.random() < 0.25,
                 transpose=kind == "resolve" and rng.random() < 0.4,
                 tol=1e-13 if kind == "autograd" else 1e-10)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

def _specs(c):
    """(MNASpec, seed) of each pattern of the case; a group's orders are
    spread over their logarithm from 1,000 (or half the largest) to n."""
    if c["kind"] != "group":
        nv = max(1, c["n"] // 125)
        return [(mna.MNASpec(n_nodes=c["n"] - nv, n_vsrc=nv, extra_lo=0, extra_hi=c["extra"], n_rails=c["rails"],
                             rail_deg=c["rail_deg"]), c["pattern"])]
    out = []
    lo, hi = math.log(min(1000, c["n"] // 2)), math.log(c["n"])
    for m in range(c["count"]):
        n = int(math.exp(lo + (hi - lo) * m / (c["count"] - 1)))
        nv = max(1, n // 125)
        out.append((mna.MNASpec(n_nodes=n - nv, n_vsrc=nv, extra_lo=0, extra_hi=c["extra"] - m % 2, n_rails=c["rails"],
                                rail_deg=max(8, n // 40)), c["pattern"] + m))
    return out


@functools.lru_cache(maxsize=2)
def _patterns(key):
    """The case's matrices and their host analyses.  A program analyses a
    circuit once and keeps the result for every later value set."""
    mats = [mna.mna_csc(spec, seed) for spec, seed in key]
    return mats, analyze_many(mats) if len(mats) > 1 else [Analysis(*mats[0])]


def _values(c, seed):
    """Host value sets and right-hand sides, made from the seed."""
    mats, _ = _patterns(tuple(_specs(c)))
    if c["kind"] == "group":
        return [(mna.perturb_values(d, 1000 * seed + m), mna.rhs(n, 1000 * seed + 500 + m))
                for m, (d, _, _, n) in enumerate(mats)]
    d, _, _, n = mats[0]
    return [(mna.perturb_values(d, 1000 * seed + m), mna.rhs(n, 1000 * seed + 500 + m)) for m in range(c["count"])]


def prepare(case, seed):
    c = case
    _, analyses = _patterns(tuple(_specs(c)))
    vals = _values(c, seed)
    plans = [Plan(a, use_graph=c["graph"]) for a in analyses]
    s = {"case": c, "plan": plans[0], "plans": plans}
    if c["kind"] == "group":
        s["group"] = Group(plans)
        s["ax"] = [torch.from_numpy(v).cuda() for v, _ in vals]
        s["b"] = [torch.from_numpy(b).cuda() for _, b in vals]
    elif c["kind"] in ("batch", "refactor"):
        s["ax"] = torch.from_numpy(np.stack([v for v, _ in vals])).cuda()
        s["b"] = torch.from_numpy(np.stack([b for _, b in vals])).cuda()
        s["lu"] = torch.empty(c["count"], plans[0].nnz_lu, dtype=torch.float32, device="cuda")
        s["x"] = torch.empty(c["count"], plans[0].n, dtype=torch.float64, device="cuda")
    else:
        s["ax"] = torch.from_numpy(vals[0][0]).cuda()
        s["b"] = torch.from_numpy(vals[0][1]).cuda()
        s["b32"] = s["b"].to(torch.float32)
        s["lu"] = torch.empty(plans[0].nnz_lu, dtype=torch.float32, device="cuda")
        s["x"] = torch.empty(plans[0].n, dtype=torch.float64, device="cuda")
        s["x32"] = torch.empty(plans[0].n, dtype=torch.float32, device="cuda")
        if c["kind"] == "resolve":
            plans[0].refresh(s["ax"], s["lu"])
            plans[0].factor(s["lu"])
        if c["kind"] == "autograd":
            s["target"] = torch.from_numpy(np.random.default_rng(7 * seed + 3).standard_normal(plans[0].n)).cuda()
    return s


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------

def run(state):
    s, c, plan = state, state["case"], state["plan"]
    kind = c["kind"]
    if kind == "newton":
        plan.refresh(s["ax"], s["lu"])
        plan.factor(s["lu"], perturb=c["perturb"])
        plan.solve(s["lu"], s["b32"], s["x32"])
        return {"lu": s["lu"], "x": s["x32"]}
    if kind == "resolve":
        return {"x": plan.solve(s["lu"], s["b32"], s["x32"], transpose=c["transpose"])}
    if kind == "refined":
        plan.refresh(s["ax"], s["lu"])
        plan.factor(s["lu"], perturb=c["perturb"])
        x, iters, eta = plan.refine(s["ax"], s["lu"], s["b"], s["x"], tol=c["tol"], maxit=20)
        return {"lu": s["lu"], "x": x, "iters": iters, "eta": eta}
    if kind == "autograd":
        v = s["ax"].detach().requires_grad_(True)
        b = s["b"].detach().requires_grad_(True)
        x = spsolve_autograd(v, b, plan, tol=c["tol"], maxit=20)
        ((x - s["target"]) ** 2).sum().backward()
        return {"x": x.detach(), "grad_values": v.grad, "grad_b": b.grad}
    if kind == "batch":
        x, lu, iters, eta = plan.batch_solve(s["ax"], s["b"], tol=c["tol"], maxit=20, perturb=c["perturb"], lu=s["lu"],
                                             x=s["x"])
        return {"lu": lu, "x": x, "iters": iters, "eta": eta}
    if kind == "refactor":
        return {"lu": plan.batch_factor(s["ax"], s["lu"], perturb=c["perturb"])}
    xs, lus, iters, eta = s["group"].solve(s["ax"], s["b"], tol=c["tol"], maxit=20, perturb=c["perturb"])
    return {"lu": lus, "x": xs, "iters": iters, "eta": eta}


# --------------------------------------------------------------------------
# what a pass cannot do without, and its result in 64 bits
# --------------------------------------------------------------------------

def work(case):
    """Inputs read once and outputs written once; the scalar updates of the
    factorization and one multiply-add per factor entry and solve."""
    c = case
    _, analyses = _patterns(tuple(_specs(c)))
    sets = 1 if c["kind"] == "group" else c["count"]
    nbytes = flops = 0
    for a in analyses:
        n, nnz, nnz_lu = a.n, a.nnz_a, a.nnz_lu
        if c["kind"] == "resolve":
            nbytes += 4 * nnz_lu + 8 * n
            flops += 2 * nnz_lu
            continue
        nbytes += sets * (8 * nnz + 4 * nnz_lu)
        flops += sets * 2 * a.updates
        if c["kind"] == "refactor":
            continue
        f64 = c["kind"] != "newton"
        nbytes += sets * (16 * n if f64 else 8 * n)
        flops += sets * (2 * nnz_lu + (2 * nnz if f64 else 0))
        if c["kind"] == "autograd":
            nbytes += 8 * nnz + 16 * n
            flops += 2 * nnz_lu + 3 * nnz
    return {"bytes": float(nbytes), "flops": float(flops)}


def exact(case, seed):
    """The solutions by dense LU in 64 bits, where that is quick (the factors
    depend on the library's own pivot order and scaling)."""
    c = case
    specs = _specs(c)
    orders = [s.n for s, _ in specs] * (1 if c["kind"] == "group" else c["count"])
    if c["kind"] == "refactor" or sum((m / 1000.0) ** 3 for m in orders) > 700 or max(orders) > 9999:
        return None
    mats = [mna.mna_csc(spec, s) for spec, s in specs]
    vals = _values(c, seed)

    def dense(k):
        _, indices, indptr, n = mats[k if c["kind"] == "group" else 0]
        a = torch.zeros(n, n, dtype=torch.float64)
        cols = np.repeat(np.arange(n), np.diff(indptr))
        a[torch.from_numpy(indices.astype(np.int64)), torch.from_numpy(cols)] = torch.from_numpy(vals[k][0])
        return a, torch.from_numpy(indices.astype(np.int64)), torch.from_numpy(cols)

    def solve(a, b):
        return torch.linalg.solve(a, b)

    if c["kind"] in ("newton", "resolve"):
        a, _, _ = dense(0)
        b = torch.from_numpy(vals[0][1]).to(torch.float32).to(torch.float64)
        x = solve(a.T.contiguous() if c["transpose"] else a, b)
        return {"x": x} if c["kind"] == "resolve" else {"lu": None, "x": x}
    if c["kind"] == "autograd":
        a, rows, cols = dense(0)
        x = solve(a, torch.from_numpy(vals[0][1]))
        target = torch.from_numpy(np.random.default_rng(7 * seed + 3).standard_normal(a.shape[0]))
        lam = solve(a.T.contiguous(), 2.0 * (x - target))
        return {"x": x, "grad_values": -lam[rows] * x[cols], "grad_b": lam}
    xs = [solve(dense(k)[0], torch.from_numpy(b)) for k, (_, b) in enumerate(vals)]
    x = xs if c["kind"] == "group" else torch.stack(xs) if c["kind"] == "batch" else xs[0]
    return {"lu": None, "x": x, "iters": None, "eta": None}
