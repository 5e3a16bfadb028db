"""CPU check of the sweeps' streams (build_sw, choose_split in glu_plan.hip):
tests/cpp/sweep_streams_check.cpp emulates them — whole orders, as those with
the vector in LDS, and split ones, under limits small enough for the patterns
here — and compares with the row-by-row solve."""

import os
import re
import shutil
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import mna_case
from test_gpu_sweeps import _case
from test_sweep_tables import BUILD, HIPCC, PKG, ROOT, _random


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    objs = [os.path.join(BUILD, f) for f in sorted(os.listdir(BUILD))
            if f.startswith("host_") or f == "glu_kernels.o"] if os.path.isdir(BUILD) else []
    if not os.path.exists(HIPCC) or not any(o.endswith("glu_kernels.o") for o in objs):
        pytest.skip("hipcc or the library's objects are missing (run __graft_entry__.build())")
    d = tmp_path_factory.mktemp("streams")
    obj, exe = str(d / "check.o"), str(d / "check")
    flags = ["-O2", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950", "-w",
             "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc")]
    subprocess.check_call([HIPCC, *flags, "-c", os.path.join(ROOT, "tests", "cpp", "sweep_streams_check.cpp"),
                           "-o", obj])
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", obj, *objs, "-o", exe])
    yield exe
    shutil.rmtree(d, ignore_errors=True)


def _pattern(case):
    if case.startswith("rand"):
        return _random(int(case[4:]))
    if case == "edges":   # rows at every change of shape
        return _case(700, (6, 7, 16, 17, 32, 33, 64, 65, 127, 128, 129, 320, 321, 385), 777)
    if case == "long":
        return _case(2049, (1000, 1500, 449, 511, 513), 2126)
    if case == "one":
        return _case(1, (), 1)
    if case == "mesh":   # 18 x 18 x 18
        one, side = sp.identity(18), sp.diags([-1, -1], [-1, 1], (18, 18))
        line = sp.diags([-1, 6, -1], [-1, 0, 1], (18, 18))
        A = sp.csc_matrix(sp.kron(sp.kron(one, one), line) + sp.kron(sp.kron(one, side), one) +
                          sp.kron(sp.kron(side, one), one))
        A.sort_indices()
        return A.data, A.indices.astype(np.int32), A.indptr.astype(np.int32), A.shape[0]
    if case == "blocks":   # 10 dense ones
        A = sp.csc_matrix(sp.block_diag([np.ones((300, 300)) + 300 * np.identity(300)] * 10))
        A.sort_indices()
        return A.data, A.indices.astype(np.int32), A.indptr.astype(np.int32), A.shape[0]
    return mna_case(case)


def _check(checker, tmp_path, case, cap, waves):
    from pyglu.analysis import Analysis
    an = Analysis(*_pattern(case))
    path = tmp_path / "pattern.bin"
    with open(path, "wb") as f:
        for k in ("sym_c_ptr", "sym_r_idx", "l_col_ptr", "csr_r_ptr", "csr_c_idx", "csr_diag_ptr"):
            a = np.ascontiguousarray(getattr(an, k)).astype(np.uint32)
            f.write(np.uint64(a.size).tobytes())
            f.write(a.tobytes())
    r = subprocess.run([checker, str(path), str(cap), str(waves)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("case", ["one", "edges", "long", "mna600", "mna2k", "small", "add32", "rand0", "rand1", "rand2"])
@pytest.mark.parametrize("waves", [1, 4, 16])
def test_whole_orders(checker, tmp_path, case, waves):
    assert "bit for bit" in _check(checker, tmp_path, case, 0, waves)


@pytest.mark.parametrize("case,most", [("mesh", 1.1), ("blocks", 1.2)])
def test_no_wave_is_waited_for(checker, tmp_path, case, most):
    """A step lasts as long as the wave with the most chunks in it takes: few
    steps beyond the share of every wave, rows of several chunks (which have
    waves of their own) or not."""
    out = _check(checker, tmp_path, case, 0, 16)
    waited, least = map(int, re.search(r"waited for: (\d+) of at least (\d+)", out).groups())
    assert least <= waited <= most * least


@pytest.mark.parametrize("case,cap", [("mna2k", 300), ("mna2k", 1000), ("small", 700), ("small", 2500), ("batch", 4000),
                                      ("grad", 10000), ("grad", 38000)])
@pytest.mark.parametrize("waves", [4, 16])
def test_split_orders(checker, tmp_path, case, cap, waves):
    """Head parts and tail within the rows a workgroup holds."""
    out = _check(checker, tmp_path, case, cap, waves)
    assert "bit for bit" in out and int(re.search(r"parts=(\d+)", out)[1]) > 0
