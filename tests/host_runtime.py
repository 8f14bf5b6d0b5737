"""Runs Python code against libgpe_hip.so on the host runtime of
tests/drivers/host_runtime.cpp: a child process, so that the runtime's place is
taken there only.  `H` and `E` are in the code's scope."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PRELUDE = """
import ctypes, sys
import numpy as np
sys.path.insert(0, {root!r})
H = ctypes.CDLL({lib!r}, ctypes.RTLD_GLOBAL)
H.hh_launches.restype = ctypes.c_char_p
H.hh_used.restype = ctypes.c_size_t
H.hh_memory.argtypes, H.hh_cost.argtypes = [ctypes.c_size_t], [ctypes.c_char_p, ctypes.c_double]
H.hh_uploaded.restype = ctypes.c_long
H.hh_fail.argtypes = [ctypes.c_long, ctypes.c_long]
from libcugpe_amd import engine as E

def launched(call, *args):
    "names of the kernels a call launches"
    H.hh_reset()
    call(*args)
    return H.hh_launches().decode().split()
"""


def build(tmp):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no C++ compiler")
    out = os.path.join(str(tmp), "libhost_runtime.so")
    subprocess.check_call([cxx, "-std=c++17", "-O1", "-shared", "-fPIC",
                           os.path.join(ROOT, "tests", "drivers", "host_runtime.cpp"), "-o", out])
    return out


def run(lib, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE.format(root=ROOT, lib=lib) + code], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:]
    return r.stdout
