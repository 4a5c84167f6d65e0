"""Contexts and transfers on a device with no room left (hipMalloc is made to
refuse, in a process of its own): the same results, bit for bit."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
BODY = """
import ctypes, sys
sys.path[:0] = [%r, %r]
shim = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
import numpy as np
from fd23_amd import _lib
_lib.load()
path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
ctypes.c_void_p.in_dll(shim, "real").value = ctypes.cast(ctypes.CDLL(path).hipMalloc, ctypes.c_void_p).value
room = ctypes.c_long.in_dll(shim, "room")
from fd23_amd.core import Context
from helpers import Problem

plain = Context.set_material
def starved(self, arrays):
    room.value = 0
    plain(self, arrays)
    room.value = -1

def results(p, storage, limit, short):
    Context.set_material = starved if limit else plain
    with p.context(storage=storage) as c:
        first = c.tile
        if limit:
            room.value = 1 << 20
        c.run(0, 9, 1)
        assert limit == (c.tile != first) or not short, (first, c.tile)
        if limit:
            room.value = 0
        names = ("U", "W", "Txx", "Txz", "Tzz") if c.wave == _lib.WAVE_PSV else ("V", "Tx", "Tz")
        out = [c.get_state(s) for s in (0, p.nshots - 1)] + [c.field(n, 0).tobytes() for n in names]
        out += [c.seismograms(s, k, 9).tobytes() for s in (0, p.nshots - 1) for k in range(c.ncomp)]
        out += [c.material(i).tobytes() for i in range(3)]
        c.set_state(out[0], p.nshots - 1)
        c.set_field(names[0], np.asarray(c.field(names[0], 0) * 2), 0)
        out += [c.get_state(s) for s in (0, p.nshots - 1)]
    room.value = -1
    return out

# shapes that need the second set, and some that do not; rows and checkpoints
# beyond the 64 KiB that a context keeps
for wave, nx, nz, shots, storage, short in (
        (_lib.WAVE_PSV, 1250, 800, 10, _lib.STORE_F32, True), (_lib.WAVE_PSV, 1250, 800, 20, _lib.STORE_F16, True),
        (_lib.WAVE_SH, 1400, 900, 3, _lib.STORE_F32, True), (_lib.WAVE_SH, 400, 200, 1, _lib.STORE_F32, True),
        (_lib.WAVE_PSV, 20000, 40, 1, _lib.STORE_BF16, False), (_lib.WAVE_PSV, 9000, 60, 2, _lib.STORE_F64, False),
        (_lib.WAVE_SH, 17000, 33, 2, _lib.STORE_F16, False)):
    kind = _lib.SRC_FORCE if wave == _lib.WAVE_SH else _lib.SRC_LINE
    p = Problem(wave, nx, nz, 8, 10.0, 7e-4, 9, seed=nx, kind=kind, rec_z=3,
                sources=[(20 + (k * (nx - 40)) // shots, 8) for k in range(shots)],
                f64=storage == _lib.STORE_F64 and wave == _lib.WAVE_PSV)
    print("case", wave, nx, nz, shots, storage, flush=True)
    a, b = (results(p, storage, limit, short) for limit in (False, True))
    assert any(a[0]) and a == b, [x == y for x, y in zip(a, b)]
"""


def test_no_room(tmp_path):
    so = str(tmp_path / "hiproom.so")
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", os.path.join(HERE, "hiproom.c"), "-o", so])
    r = subprocess.run([sys.executable, "-c", BODY % (os.path.dirname(HERE), HERE, so)], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=110)
    print(r.stdout, flush=True)
    assert r.returncode == 0, r.stdout
