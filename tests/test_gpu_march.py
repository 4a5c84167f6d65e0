"""The marching P-SV step (two steps per launch over the grid's interior, the
two passes on the frame around it) against the two-pass loop: the same
arithmetic per cell, so states, seismograms and scales are equal bit for bit.
"""
import numpy as np
import pytest

from fd23_amd import _lib
from helpers import Problem

pytestmark = pytest.mark.gpu

REACH, TX, TZ, OWN = 12, 64, 16, 224  # cells of recomputation, tile, owned columns of a strip


def march_tile():
    lib = _lib.load()
    import ctypes
    for t in range(lib.fd23_num_tiles()):
        v = [ctypes.c_int() for _ in range(4)]
        _lib.check(lib.fd23_tile_shape(t, *(ctypes.byref(x) for x in v)))
        if lib.fd23_tile_kind(t) == _lib.TILE_FUSED and v[3].value == -1:
            return t
    raise AssertionError("no marching shape")


def rectangle(nx, nz, npml, top):
    lo = max(npml, 4) + REACH
    ztop = lo if top else 4 + REACH
    return (-(-lo // TX) * TX, (nx - lo) // TX * TX, -(-ztop // TZ) * TZ, (nz - lo) // TZ * TZ)


# nx, nz, npml, topabsorb, shots: the smallest rectangle (one tile), one cell
# less (none), a second strip of 96 columns, exactly one strip, an absorbing
# top, enough shots for segments of several tens of rows
GRIDS = [(145, 49, 5, False, 1), (144, 49, 5, False, 1), (404, 97, 5, False, 2), (448, 131, 20, True, 2),
         (300, 220, 12, False, 3), (420, 150, 8, True, 40)]


@pytest.mark.parametrize("storage", [_lib.STORE_F32, _lib.STORE_F16, _lib.STORE_BF16, _lib.STORE_F64])
@pytest.mark.parametrize("nx,nz,npml,top,shots", GRIDS)
def test_march_equals_two_passes(nx, nz, npml, top, shots, storage):
    if shots > 4 and storage == _lib.STORE_F64:
        pytest.skip("FP64 runs the two passes: the small grids show it")
    x0, x1, z0, z1 = rectangle(nx, nz, npml, top)
    rng = np.random.default_rng(nx + nz)
    # sources at the rectangle's corners and edges, on strip edges, inside,
    # in the frame; the P kind spreads over three columns and two rows
    spots = [(x0, z0), (x1 - 1, z1 - 1), (min(x0 + OWN, nx - npml - 2), (z0 + z1) // 2), (x0 - 1, z0 - 1),
             (nx // 2, 6 + (npml if top else 0)), (x0 + 1, z0 + 17)]
    srcs = [spots[k % len(spots)] for k in range(shots)]
    kind = _lib.SRC_P if nx % 4 == 0 else _lib.SRC_LINE
    p = Problem(_lib.WAVE_PSV, nx, nz, npml, 10.0, 7e-4, 180, seed=nx, topabsorb=top, kind=kind, sources=srcs,
                rec_z=npml + 3 if top else 2, f64=storage == _lib.STORE_F64)
    more_x = np.concatenate([[x0 - 1, x0, x1 - 1, min(x1, nx - 1), x0 + OWN - 1, min(x0 + OWN, nx - 1), 0, nx - 1],
                             rng.integers(0, nx, 600)])
    more_z = np.concatenate([[z0, z0 - 1, z1 - 1, min(z1, nz - 1), z0 + 15, z0 + 16, nz - 1, 0],
                             rng.integers(0, nz, 300), np.full(300, (z0 + z1) // 2)])
    p.rx = np.concatenate([p.rx, np.clip(more_x, 0, nx - 1)]).astype(np.int32)
    p.rz = np.concatenate([p.rz, np.clip(more_z, 0, nz - 1)]).astype(np.int32)

    def run(tile):
        with p.context(storage=storage) as ctx:
            ctx.tile = tile
            ctx.run(0, 131, 3)       # a chunk of 128 steps, one pair and a single step
            ctx.run(131, 1, 3)
            ctx.run(132, 27, 3)      # pairs and a single step
            for it in range(159, 162):
                ctx.step_stress()
                ctx.inject(it)
                ctx.step_velocity()
                ctx.record(it, 3)
            ctx.run(162, 18, 3)
            ctx.sync()
            state = [ctx.get_state(s) for s in range(shots)]
            seis = [ctx.seismograms(s, c, 60) for s in range(shots) for c in range(2)]
            return state, seis, ctx.get_scales(13)

    want, got = run(0), run(march_tile())
    assert all(np.isfinite(x).all() for x in want[1]) and any(np.abs(x).max() > 0 for x in want[1])
    for k in range(13):
        assert want[2][0][k] == got[2][0][k] and want[2][1][k] == got[2][1][k], k
    for s in range(shots):
        assert want[0][s] == got[0][s], s
    for a, b in zip(want[1], got[1]):
        assert np.array_equal(a, b)


def test_march_leaves_idle_slots_and_windows_to_the_passes():
    """An idle slot keeps its fields, and a first-arrival window applies, on a
    context set to the marching shape."""
    nx, nz = 256, 128
    p = Problem(_lib.WAVE_PSV, nx, nz, 8, 10.0, 7e-4, 60, seed=4, sources=[(100, 30), (120, 40)], rec_z=20)
    with p.context() as ctx, p.context() as ref:
        ctx.tile = march_tile()
        ref.tile = 0
        for c in (ctx, ref):
            c.run(0, 30, 1)
            c.set_shot_slot(1, active=False)
            c.run(30, 11, 1)
            c.sync()
        for s in range(2):
            assert ctx.get_state(s) == ref.get_state(s)
    z, x = np.mgrid[0:nz, 0:nx]
    times = (np.hypot(x - 100, z - 30) * 10.0 / 6000.0).astype(np.float32)
    with p.context() as ctx, p.context() as ref:
        ctx.tile = march_tile()
        ref.tile = 0
        for c in (ctx, ref):
            c.set_punch(times, 0.005, 0.02, 7e-4)
            c.run(0, 41, 1)
            c.sync()
        assert ctx.get_state(0) == ref.get_state(0)
