"""Runs a piece of Python in a process of its own on top of fake_hip.cpp: `F` is its interface, host code of the library runs unchanged, launches run
nothing."""
import functools
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
HEAD = """
import ctypes as C, sys
F = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
F.fake_live.restype = F.fake_peak.restype = C.c_size_t
F.fake_limit.argtypes = [C.c_size_t]
count = lambda name: F.fake_count(name.encode())
sys.path[:0] = [sys.argv[2], sys.argv[3]]
"""


@functools.lru_cache(None)
def library():
    so = os.path.join(tempfile.mkdtemp(prefix="fake_hip"), "fake_hip.so")
    subprocess.check_call(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", "-w", "-I/opt/rocm/include", "-o", so, os.path.join(HERE, "fake_hip.cpp")])
    return so


def run(code, timeout=100):
    env = {k: v for k, v in os.environ.items() if not k.startswith("PI_")}
    r = subprocess.run([sys.executable, "-c", HEAD + code, library(), os.path.dirname(HERE), HERE], capture_output=True, text=True, timeout=timeout, env=env)
    assert r.returncode == 0, r.stderr[-1500:]
    return r.stdout
