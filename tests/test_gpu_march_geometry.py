"""The marching steps at the edges of their real geometry (the rectangle, its
strips of 224 or 480 columns and its segments) against the two-pass loop, from
random fields in every cell, bit for bit."""
import numpy as np
import pytest

from fd23_amd import _lib
from helpers import Problem
from test_gpu_march import march_tile

pytestmark = pytest.mark.gpu

REACH, TAIL = 12, 24


def up(a, n):
    return -(-a // n) * n


def rectangle(nx, nz, npml, top, deep=10 ** 6):
    """The library's marching rectangle, or None; deep: the deepest of the
    source's reach and the receiver rows."""
    lo = max(npml, 4) + REACH
    x0, x1 = up(lo, 16), max(nx - lo, 0) // 16 * 16
    z0, z1 = up(lo if top else 4 + REACH, 16), max(nz - lo, 0) // 16 * 16
    if x1 <= x0 or z1 <= z0:
        return None
    below = up(max(deep, z0 - 1) + 1, 16)
    return (x0, x1, below if below - z0 <= (z1 - z0) // 8 else z0, z1)


def strips(rect, shots):
    """Columns of a strip with its halo, and rows of a segment."""
    x0, x1, z0, z1 = rect
    best = None
    for W in (256, 512):
        columns, slots = -(-(x1 - x0) // (W - 32)) * shots, 262144 // W
        for H in range(up(z1 - z0, 8), 15, -8):
            cost = -(-columns * -(-(z1 - z0) // H) // slots) * (H + TAIL)
            if best is None or cost < best[0]:
                best = (cost, W, H)
    return best[1:]


# nx, nz, npml, topabsorb, shots, and what march_work makes of it: (W, H), or
# None without a rectangle
GRIDS = [(65, 49, 5, False, 1, (256, 16)),      # one block of 16 x 16 cells
         (64, 49, 5, False, 1, None),           # a column less
         (65, 48, 5, False, 1, None),           # a row less
         (520, 150, 8, True, 3, (256, 16)),     # strips of 224, 224 and 16 columns
         (548, 100, 8, False, 114, (256, 32)),  # segments of several eights of rows
         (512, 180, 8, True, 171, (256, 64)),
         (1025, 101, 8, False, 52, (512, 16)),  # 512 columns: two full strips of 480
         (530, 100, 8, False, 140, (512, 24))]  # one strip
KINDS = [(_lib.WAVE_PSV, _lib.STORE_F32), (_lib.WAVE_PSV, _lib.STORE_F16), (_lib.WAVE_PSV, _lib.STORE_BF16),
         (_lib.WAVE_SH, _lib.STORE_F32)]


def compare(p, storage):
    names = ("U", "W", "Txx", "Tzz", "Txz") if p.wave == _lib.WAVE_PSV else ("V", "Tx", "Tz")
    shots = sorted({0, 1 % p.nshots, p.nshots - 1})
    out = []
    for tile in (0, march_tile()):
        with p.context(storage=storage, max_frames=16) as ctx:
            ctx.tile = tile
            ctx.run(0, 0, 1)  # the scales of 16-bit storage come with the first run
            scaled = storage in (_lib.STORE_F16, _lib.STORE_BF16)
            sc = ctx.get_scales(5)[0] * 64.0 if scaled else np.full(5, 1e-2)
            rng = np.random.default_rng(p.nx)
            for s in shots:
                for i, f in enumerate(names):
                    vel = len(f) == 1
                    amp = sc[0 if vel else 2] if scaled else sc[0] * (float(p.mat[0].max()) if vel else 1.0)
                    ctx.set_field(f, (amp * rng.standard_normal((p.nz, p.nx))).astype(np.float32), s)
            ctx.run(0, 19, 3)  # pairs and a single step
            ctx.run(19, 12, 3)
            ctx.sync()
            out.append([ctx.get_state(s) for s in shots] +
                       [ctx.seismograms(s, c, 11).tobytes() for s in shots for c in range(ctx.ncomp)])
    for a in out[0][:len(shots)]:
        v = np.frombuffer(a, np.float32)
        assert np.isfinite(v).all() and (v != 0).mean() > 0.5
    for i, (a, b) in enumerate(zip(*out)):
        assert a == b, i


@pytest.mark.parametrize("wave,storage", KINDS)
@pytest.mark.parametrize("nx,nz,npml,top,shots,shape", GRIDS)
def test_rectangle_strips_and_segments(nx, nz, npml, top, shots, shape, wave, storage):
    rect = rectangle(nx, nz, npml, top)
    assert (rect and strips(rect, shots)) == shape
    x0, x1, z0, z1 = rect or (32, 48, 16, 32)
    W, H = shape or (256, 16)
    own = W - 32
    # around every strip and segment edge, the rectangle's corners, the halos
    # of 12 cells and of 16 columns
    cols = sorted({min(max(x + d, 2), nx - 3) for x in [*range(x0, x1, own), x1] for d in (-16, -13, -12, -1, 0, 1, 15)})
    rows = sorted({min(max(z + d, 2), nz - 3) for z in [*range(z0, z1, H), z1] for d in (-13, -12, -1, 0, 7, 8)})
    srcs = [(cols[(3 * k) % len(cols)], rows[(5 * k + 1) % len(rows)]) for k in range(shots)]
    kind = _lib.SRC_P if nx % 2 else _lib.SRC_FORCE if wave == _lib.WAVE_SH else _lib.SRC_LINE
    p = Problem(wave, nx, nz, npml, 10.0, 7e-4, 40, seed=nx, topabsorb=top, kind=kind, sources=srcs)
    x, z = np.meshgrid(cols, rows)
    p.rx, p.rz = x.ravel().astype(np.int32), z.ravel().astype(np.int32)
    compare(p, storage)


@pytest.mark.parametrize("wave,storage", KINDS)
@pytest.mark.parametrize("zs,first", [(17, 32), (18, 32), (19, 16)])
def test_shallow_events_move_the_rectangle(zs, first, wave, storage):
    """The rectangle starts below shallow events while that costs it an eighth
    of its rows at most."""
    nx, nz, npml = 320, 161, 5
    deep = zs + 1 + REACH
    assert rectangle(nx, nz, npml, False, deep) == (32, 288, first, 144)
    kind = _lib.SRC_FORCE if wave == _lib.WAVE_SH else _lib.SRC_P
    p = Problem(wave, nx, nz, npml, 10.0, 7e-4, 40, seed=zs, kind=kind, sources=[(32, zs), (257, 3)])
    p.rx = np.arange(nx, dtype=np.int32)
    p.rz = np.where(p.rx % 2, deep, 15).astype(np.int32)
    compare(p, storage)
