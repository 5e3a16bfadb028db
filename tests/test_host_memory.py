"""Host memory running out inside a C entry point: a status code, never a C++
exception through it (which would end the process)."""

import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("count", [20_000_000, 2_000_000_000])
def test_group_larger_than_memory(count):
    """A group whose host tables exceed the process's memory limit."""
    code = f"""
import sys, resource, ctypes as C
sys.path.insert(0, {os.path.join(ROOT, 'glu-hcu_amd')!r})
from pyglu import _capi
L = _capi.lib()
used = int(open('/proc/self/statm').read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (1 << 30), used + (1 << 30)))
plans, g = (C.c_void_p * 1)(), C.c_void_p()
status = L.glu_group_create(plans, {count}, C.byref(g))
print('status', status, L.glu_last_error().decode(), flush=True)
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr[-500:])
    assert "status -3" in r.stdout
