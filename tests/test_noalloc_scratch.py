"""CPU check of glu_refine_noalloc's scratch layout: no order within its limit
is refused (tests/cpp/scratch_check.cpp)."""

import os
import subprocess

import pytest

from test_sweep_tables import BUILD, HIPCC, PKG, ROOT


def test_every_order_within_the_limit_fits(tmp_path):
    objs = [os.path.join(BUILD, f) for f in sorted(os.listdir(BUILD))
            if f.startswith("host_") or f == "glu_kernels.o"] if os.path.isdir(BUILD) else []
    if not os.path.exists(HIPCC) or not any(o.endswith("glu_kernels.o") for o in objs):
        pytest.skip("hipcc or the library's objects are missing (run __graft_entry__.build())")
    obj, exe = str(tmp_path / "check.o"), str(tmp_path / "check")
    flags = ["-O2", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950", "-w",
             "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc")]
    subprocess.check_call([HIPCC, *flags, "-c", os.path.join(ROOT, "tests", "cpp", "scratch_check.cpp"), "-o", obj])
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", obj, *objs, "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
