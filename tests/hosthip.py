"""Runs a piece of Python against libfd23.so with the HIP runtime replaced by
hosthip.c, in a process of its own."""
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
SETUP = """
import ctypes, sys
sys.path[:0] = [%r, %r]
hip = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
class Hip:
    def __getattr__(self, n):
        return (ctypes.c_int if n == "hh_error" else ctypes.c_long).in_dll(hip, n).value
    def __setattr__(self, n, v):
        (ctypes.c_int if n == "hh_error" else ctypes.c_long).in_dll(hip, n).value = v
hh = Hip()
import numpy as np
from fd23_amd import _lib, host
from fd23_amd.core import Context
PSV, SH = _lib.WAVE_PSV, _lib.WAVE_SH
F32, F16, BF16, F64 = _lib.STORE_F32, _lib.STORE_F16, _lib.STORE_BF16, _lib.STORE_F64
def context(wave, nx, nz, shots=1, storage=F32, npml=8, zs=8, zr=4, nt=16):
    c = Context(wave, nx, nz, npml, nshots=shots, storage=storage, max_frames=nt, max_rec=nx)
    a = np.ones((nz, nx), c.cdtype)
    c.set_material([a] * (5 if wave == PSV else 3))
    c.set_cpml(host.cpml_pack(wave, nx, nz, npml, 1e-3, 1e-6, 300.0, 10.0))
    for s in range(shots):
        c.set_source(s, _lib.SRC_LINE, nx // 2, zs, np.ones(4), np.ones(3))
        for k in range(c.ncomp):
            c.set_receivers(s, k, np.arange(nx, dtype=np.int32), np.full(nx, zr, np.int32))
    return c
def raises(code, f, *a):
    try:
        f(*a)
    except _lib.Fd23Error as e:
        assert code in str(e), e
    else:
        raise AssertionError("no error: " + code)
"""


def run(body):
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "hosthip.so")
        subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-w", os.path.join(HERE, "hosthip.c"), "-o", so])
        r = subprocess.run([sys.executable, "-c", SETUP % (os.path.dirname(HERE), HERE, so) + body],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    return r.stdout
