"""What sources and receivers inside the marching step's rectangle cost: a run
with them against the same run with all of them near the surface, where the
frame takes them.  The bounds lie between what the loop with events costs by
itself (5 to 25%) and what a list read one entry after another, or stresses
kept in scratch memory, made of it (1.4 to 1.9 times)."""
import time

import numpy as np
import pytest

from fd23_amd import _lib, host
from fd23_amd.core import Context
from test_gpu_march import march_tile

pytestmark = pytest.mark.gpu


def seconds(wave, nx, nz, shots, storage, zs, zr, nt=32):
    with Context(wave, nx, nz, 20, nshots=shots, storage=storage, max_frames=nt, max_rec=nx) as ctx:
        nv, nm = (2, 5) if wave == _lib.WAVE_PSV else (1, 3)
        ctx.set_material([np.full((nz, nx), 1e-4 if i < nv else 500.0, np.float32) for i in range(nm)])
        ctx.set_cpml(host.cpml_pack(wave, nx, nz, 20, 1e-3, 1e-6, 300.0, 10.0))
        stf, M = host.ricker(nt, 1e-3, 30.0), np.array([1.0, 0.3, 1.0])
        rx, rz = np.arange(nx, dtype=np.int32), np.full(nx, zr, np.int32)
        for s in range(shots):
            ctx.set_source(s, _lib.SRC_LINE, nx // 2, zs, stf, M)
            for c in range(ctx.ncomp):
                ctx.set_receivers(s, c, rx, rz)
        ctx.tile = march_tile()
        ctx.prepare(nt)
        best = 1e9
        for _ in range(8):
            ctx.sync()
            t = time.perf_counter()
            ctx.run(0, nt, 1)
            ctx.sync()
            best = min(best, time.perf_counter() - t)
        return best


# a list read entry by entry: 1.77 and 1.59 times
@pytest.mark.parametrize("wave,shots,bound", [(_lib.WAVE_PSV, 2, 1.55), (_lib.WAVE_SH, 1, 1.3)])
def test_receiver_line_at_depth(wave, shots, bound):
    nx, nz = 3000, 1800
    near = seconds(wave, nx, nz, shots, _lib.STORE_F32, 8, 4)
    deep = seconds(wave, nx, nz, shots, _lib.STORE_F32, 8, nz // 2)
    print("receiver line at depth", deep / near, flush=True)
    assert deep < bound * near


# stresses in scratch memory: 1.37 times
def test_source_at_depth():
    nx, nz = 3000, 1800
    near = seconds(_lib.WAVE_PSV, nx, nz, 2, _lib.STORE_F32, 8, 4)
    deep = seconds(_lib.WAVE_PSV, nx, nz, 2, _lib.STORE_F32, nz // 2, 4)
    print("source at depth", deep / near, flush=True)
    assert deep < 1.22 * near


# maxima gathered on every step: 1.52 and 1.49 times
@pytest.mark.parametrize("storage", [_lib.STORE_F16, _lib.STORE_BF16])
def test_source_at_depth_in_16_bits(storage):
    nx, nz = 3000, 1800
    near = seconds(_lib.WAVE_PSV, nx, nz, 4, storage, 8, 4)
    deep = seconds(_lib.WAVE_PSV, nx, nz, 4, storage, nz // 2, 4)
    print("source at depth", storage, deep / near, flush=True)
    assert deep < 1.38 * near
