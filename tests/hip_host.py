"""Runs a piece of Python against the library on hip_host.cpp's runtime (host
memory, a limit on its bytes, no kernels), in a process of its own: the
runtime's names have to be there before the library is loaded."""
import functools
import os
import subprocess
import sys
import tempfile

from product_util import PKG, ROOT

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
import numpy as np
H = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
H.hh_limit.argtypes = [ctypes.c_size_t]
H.hh_used.restype = ctypes.c_size_t
for f in ("hh_bad", "hh_captures", "hh_launches"):
    getattr(H, f).restype = ctypes.c_longlong
NO_LIMIT = (1 << 64) - 1
sys.path.insert(0, %r)
from product_util import adaptive_forest, glhip, initial_state
G = glhip()
"""


@functools.lru_cache(maxsize=None)
def _runtime():
    d = tempfile.TemporaryDirectory(prefix="hip_host")
    so = os.path.join(d.name, "libhip_host.so")
    cmd = ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wno-return-type-c-linkage", "-D__HIP_PLATFORM_AMD__",
           "-I/opt/rocm/include", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc"),
           os.path.join(HERE, "hip_host.cpp"), "-o", so]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return d, so


def run(code, timeout=300):
    """stdout of the code's process; the test fails if that does."""
    _, so = _runtime()
    r = subprocess.run([sys.executable, "-c", PRELUDE % (so, HERE) + code], capture_output=True, text=True,
                       timeout=timeout)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-4000:])
    return r.stdout
