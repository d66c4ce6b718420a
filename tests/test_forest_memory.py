"""A forest of millions of one-node trees is taken with memory in proportion to
its nodes: with 3 GB of address space to spare, the entry point returns (without
a GPU: its status says so) instead of ending the process in an allocation."""

import subprocess
import sys

import pytest

from tests.conftest import ROOT, have_gpu

CODE = """
import ctypes, resource
import numpy as np
from fd_adi_amd import _lib
n = 6000000
start = np.arange(n + 1, dtype=np.int64)
i32, u8, f8 = np.zeros(n, np.int32), np.ones(n, np.uint8), np.zeros(n)
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (3 << 30), resource.RLIM_INFINITY))
h = ctypes.c_void_p()
st = _lib.lib.fdadi_forest_create(n, _lib.ptr(start), 3, _lib.ptr(i32), _lib.ptr(f8),
                                  _lib.ptr(i32), _lib.ptr(i32), _lib.ptr(u8), _lib.ptr(f8), 0.0,
                                  ctypes.byref(h))
print("status", st)
"""


def test_many_tiny_trees():
    if have_gpu():
        pytest.skip("the limit would also bound the HIP runtime's own reservations")
    r = subprocess.run([sys.executable, "-c", CODE], cwd=ROOT, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0 and "status" in r.stdout, (r.returncode, r.stderr[-500:])
