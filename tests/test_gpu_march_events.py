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


def context(wave, nx, nz, shots, storage, zs, rx, rz, nt):
    ctx = Context(wave, nx, nz, 20, nshots=shots, storage=storage, max_frames=nt, max_rec=len(rx))
    nv, nm = (2, 5) if wave == _lib.WAVE_PSV else (1, 3)
    ctx.set_material([np.full((nz, nx), 1e-4 if i < nv else 500.0, np.float32) for i in range(nm)])
    ctx.set_cpml(host.cpml_pack(wave, nx, nz, 20, 1e-3, 1e-6, 300.0, 10.0))
    stf, M = host.ricker(nt, 1e-3, 30.0), np.array([1.0, 0.3, 1.0])
    for s in range(shots):
        ctx.set_source(s, _lib.SRC_LINE, nx // 2, zs, stf, M)
        for c in range(ctx.ncomp):
            ctx.set_receivers(s, c, np.asarray(rx, np.int32), np.asarray(rz, np.int32))
    return ctx


def run_seconds(ctx, nt):
    ctx.prepare(nt)
    best = 1e9
    for _ in range(8):
        ctx.sync()
        t = time.perf_counter()
        ctx.run(0, nt, 1)
        ctx.sync()
        best = min(best, time.perf_counter() - t)
    return best


def seconds(wave, nx, nz, shots, storage, zs, zr, nt=32):
    with context(wave, nx, nz, shots, storage, zs, np.arange(nx), np.full(nx, zr), nt) as ctx:
        ctx.tile = march_tile()
        return run_seconds(ctx, nt)


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


def test_tuning_sees_the_events():
    """A borehole of receivers makes the marching step 1.25 times as slow as the
    best passes here, with no event inside it is as fast."""
    nx, nz, nt = 1400, 900, 32
    with context(_lib.WAVE_PSV, nx, nz, 16, _lib.STORE_F16, 8, np.full(nz - 8, nx // 2), np.arange(4, nz - 4), nt) as ctx:
        ctx.tile = 1
        passes = run_seconds(ctx, nt)
        tile, _ = ctx.autotune(8)
        tuned = run_seconds(ctx, nt)
        print("tuned with a borehole", tile, tuned / passes, flush=True)
        assert tuned < 1.12 * passes
