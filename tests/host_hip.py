"""Runs a piece of Python against the library on the stand-in runtime of
host_hip.cpp (no GPU, kernels do not run), in a process of its own so that the
stand-in's symbols come before the runtime's."""
import functools
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
hh = C.CDLL({shim!r}, mode=C.RTLD_GLOBAL)
hh.hh_log.restype = C.c_char_p
hh.hh_limit.argtypes = [C.c_size_t]
hh.hh_held.restype = C.c_size_t
hh.hh_allow.argtypes = [C.c_long]
def log():
    return [l.split() for l in hh.hh_log().decode().splitlines()]
def launched(name):
    return sum(1 for l in log() if l[0] == "launch" and name in l[1])
import numpy as np
import elvibrot_amd as E
def dev(n):
    p = C.c_void_p()
    assert hh.hipMalloc(C.byref(p), C.c_size_t(8 * n)) == 0
    return p
"""


@functools.lru_cache(maxsize=1)
def _shim():
    so = os.path.join(tempfile.mkdtemp(prefix="host_hip_"), "host_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", so, os.path.join(HERE, "host_hip.cpp")], check=True)
    return so


def run(code):
    pre = PRELUDE.format(root=os.path.dirname(HERE), shim=_shim())
    r = subprocess.run([sys.executable, "-c", pre + code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
