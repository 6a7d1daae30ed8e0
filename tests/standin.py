"""The library on a stand-in HIP runtime (tests/cpp/hip_standin.cpp): its host
side without a GPU. `run` executes a piece of Python in a process of its own,
where `hip` is the stand-in and `av` and `W` are the package; kernels do
nothing there, so only what the host keeps can be tested."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, sys
import numpy as np
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
for f in ("standin_failures_left", "standin_stale", "standin_launches", "standin_captures", "standin_live"):
    getattr(hip, f).restype = C.c_long
hip.standin_fail_after.argtypes = [C.c_long]
sys.path.insert(0, sys.argv[2])
import atomiverse_amd as av
from atomiverse_amd import workloads as W

def live():
    sizes = np.zeros(65536, np.int64)
    n = hip.standin_live(sizes.ctypes.data_as(C.c_void_p), C.c_long(sizes.size))
    return sizes[:n].tolist()

def make(ctx, w):
    s = av.System(ctx, w.n, w.box)
    W.upload(s, w)
    W.configure(s, w)
    return s

def failing(call):
    '''Runs `call` again and again, its first, second, ... allocation failing,
    until one run meets no failure; yields after every failed run.'''
    k = 0
    while True:
        hip.standin_fail_after(k)
        try:
            call()
        except av.HipError:
            pass
        done = hip.standin_failures_left() >= 0
        hip.standin_fail_after(-1)
        if done:
            return
        yield k
        k += 1
"""


@pytest.fixture(scope="session")
def standin(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("standin") / "hip_standin.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-o", so,
                    os.path.join(ROOT, "tests", "cpp", "hip_standin.cpp")], check=True)

    def run(code):
        out = subprocess.run([sys.executable, "-c", PRELUDE + code, so, ROOT], capture_output=True, text=True,
                             timeout=300)
        assert out.returncode == 0, out.stdout[-2000:] + out.stderr[-4000:]
        return out.stdout

    return run
