"""Child processes that load libswept1d.so with tests/hip_stub.cpp in the HIP
runtime's place (no GPU)."""
import os
import subprocess
import sys

from conftest import ROOT

TESTS = os.path.dirname(os.path.abspath(__file__))
HEAD = r'''
import ctypes as C, importlib, sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[2]]
sw = importlib.import_module("1dsweptcuda_amd")
stub = C.CDLL(None)
sw.lib()
def ks(n, count=1):
    return np.ones(count, np.int32), np.full(count, n, np.int64), np.full(count, 0.005), np.full(count, 0.5)
def raises(f, code):
    try:
        f()
    except sw.SweptError as e:
        assert "(%d)" % code in str(e), e
        return
    raise AssertionError("no error")
EINVAL, EDEVICE, ENOMEM = -1, -2, -3
'''


def build(folder):
    so = str(folder / "hip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-shared", "-fPIC", "-o", so,
                    os.path.join(TESTS, "hip_stub.cpp")], check=True)
    return so


def run(so, script):
    """Runs the script after HEAD; it ends by printing "done"."""
    preload = " ".join(p for p in (so, os.environ.get("LD_PRELOAD", "")) if p)
    r = subprocess.run([sys.executable, "-c", HEAD + script, ROOT, TESTS], env=dict(os.environ, LD_PRELOAD=preload),
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr
