"""CPU check of the factorization's window and phase streams (glu_plan.hip):
tests/cpp/factor_streams_check.cpp runs them on the host — every slot and place
in range, no two lanes of a step in each other's way, every product made and
used once — and compares with the updates in schedule order bit for bit, on the
patterns of the GPU test of the phases and under small limits of LDS."""

import os
import re
import shutil
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_phases import CASES
from test_sweep_tables import BUILD, HIPCC, PKG, ROOT


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    objs = [os.path.join(BUILD, f) for f in sorted(os.listdir(BUILD))
            if f.startswith("host_") or f == "glu_kernels.o"] if os.path.isdir(BUILD) else []
    if not os.path.exists(HIPCC) or not any(o.endswith("glu_kernels.o") for o in objs):
        pytest.skip("hipcc or the library's objects are missing (run __graft_entry__.build())")
    d = tmp_path_factory.mktemp("factor")
    obj, exe = str(d / "check.o"), str(d / "check")
    flags = ["-O2", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950", "-w",
             "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc")]
    subprocess.check_call([HIPCC, *flags, "-c", os.path.join(ROOT, "tests", "cpp", "factor_streams_check.cpp"),
                           "-o", obj])
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", obj, *objs, "-o", exe])
    yield exe
    shutil.rmtree(d, ignore_errors=True)


def _csc(A):
    A = sp.csc_matrix(A)
    A.sort_indices()
    return A.data.copy(), A.indices.astype(np.int32), A.indptr.astype(np.int32), A.shape[0]


def _mesh(m, dims):
    """Laplacian of an m x m (x m) mesh."""
    one, line = sp.identity(m), sp.diags([-1.0, 2.0, -1.0], [-1, 0, 1], (m, m))
    A = 0
    for d in range(dims):
        term = sp.identity(1)
        for k in range(dims):
            term = sp.kron(term, line if k == d else one)
        A = A + term
    return _csc(A)


# patterns whose leading steps join into few components
JOINED = {"dense": lambda: _csc(np.random.default_rng(1).uniform(0.1, 1, (300, 300)) + 300 * np.eye(300)),
          "mesh2": lambda: _mesh(110, 2), "mesh3": lambda: _mesh(13, 3),
          "blocks": lambda: _csc(sp.block_diag([np.random.default_rng(k).uniform(0.1, 1, (150, 150)) + 150 * np.eye(150)
                                                for k in range(12)]))}


@pytest.fixture(scope="module")
def pattern(tmp_path_factory):
    d = tmp_path_factory.mktemp("patterns")

    def dump(name):
        path = d / name
        if not path.exists():
            from pyglu.analysis import Analysis
            an = Analysis(*(CASES.get(name) or JOINED[name])())
            with open(path, "wb") as f:
                for k in ("sym_c_ptr", "sym_r_idx", "l_col_ptr", "csr_r_ptr", "csr_c_idx", "csr_diag_ptr",
                          "level_ptr", "level_idx"):
                    a = np.ascontiguousarray(getattr(an, k)).astype(np.uint32)
                    f.write(np.uint64(a.size).tobytes())
                    f.write(a.tobytes())
        return str(path)
    return dump


def _check(checker, path, values, bin_values, reverse=0):
    r = subprocess.run([checker, path, str(values), str(bin_values), str(reverse)], capture_output=True, text=True,
                       timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and "bit for bit" in r.stdout, r.stdout + r.stderr
    return {k: int(v) for k, v in re.findall(r"(\w+)=(\d+)", r.stdout)}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("values", [60, 700])
def test_streams(checker, pattern, name, values):
    got = _check(checker, pattern(name), values, 19000)
    # the patterns reach what they are there for: phases, and entries of one
    # product a block (32 blocks: a lane each, 33: a wave each), and of both kinds
    if name not in ("one", "few"):
        assert got["phases"]
    if values == 700 and name in ("lane", "wave"):
        assert (got["lane_entries"] > 0, got["wave_entries"] > 0) == (name == "lane", name == "wave")
    if name in ("unsym300", "mna2k", "grad"):
        assert got["lane_entries"] and got["wave_entries"]


@pytest.mark.parametrize("name", ["many", "unsym1500", "mna2k", "grad"])
@pytest.mark.parametrize("bin_values", [30, 300, 2000])
def test_bins_fit_small_limits(checker, pattern, name, bin_values):
    """Bins of a device with less LDS: none holds more values than it may."""
    assert _check(checker, pattern(name), 60, bin_values)["largest"] <= bin_values


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("values", [60, 700])
def test_levels_listed_downward(checker, pattern, name, values):
    """A caller's pattern may list a level's columns in any order: the phases
    subtract in that order too, as the other steps do."""
    _check(checker, pattern(name), values, 19000, reverse=1)


@pytest.mark.parametrize("name", list(JOINED))
@pytest.mark.parametrize("values", [700, 39800])
def test_work_of_a_phase_is_spread(checker, pattern, name, values):
    """Steps whose work would fall on a few workgroups stay launches over the
    whole card: 50 ns a chunk on the busiest bin, at most 5 us a step."""
    assert _check(checker, pattern(name), values, 19000)["busiest"] <= 100
